// Host-side building blocks shared by the engines: device buffers, the CG-product tables, MFMA fragment packing, the
// tile-GEMM job lists of the FC layers, and the stream / profiling base of an engine.
#pragma once

#include "device_mem.hpp"
#include "engine.hpp"
#include "jit_prod.hpp"
#include "kernels_1l.hpp"

#include <algorithm>
#include <atomic>
#include <functional>
#include <map>
#include <mutex>
#include <cmath>
#include <cstring>
#include <numeric>

namespace grhip {

#define HIP_CHECK(expr)                                                                                         \
  do {                                                                                                          \
    hipError_t e_ = (expr);                                                                                     \
    if (e_ != hipSuccess)                                                                                       \
      throw Error(std::string("HIP error: ") + hipGetErrorString(e_) + " in " #expr " (" __FILE__ ":" + std::to_string(__LINE__) + ")"); \
  } while (0)

// Messages of the library (choice of a chunk, retries after a failed allocation, kernels that fall back to their
// table-driven form) go to a callback the caller installs, as the reference's grace::Logger (libgrace/include/grace/
// error.h:10-15): fn(user, level, message), level 0 information, 1 warning.  Without a callback they are dropped.
typedef void (*LogCallback)(void *user, int level, const char *message);
struct LogSink {
  std::atomic<LogCallback> fn{nullptr};
  std::atomic<void *> user{nullptr};
};
inline LogSink &log_sink()
{
  static LogSink s;
  return s;
}
inline void log_message(int level, const std::string &m)
{
  const LogCallback f = log_sink().fn.load();
  if (f) f(log_sink().user.load(), level, m.c_str());
}

// pinned host memory of the engine (allocated, never registered): staging of the small per-call transfers, so that they are
// asynchronous copies on the engine's stream with one wait instead of one blocking copy each
struct PinnedBuf {
  void *p = nullptr;
  size_t bytes = 0;
  PinnedBuf() = default;
  PinnedBuf(const PinnedBuf &) = delete;
  PinnedBuf &operator=(const PinnedBuf &) = delete;
  ~PinnedBuf() { release(); }
  void release()
  {
    if (p) (void) hipHostFree(p);
    p = nullptr;
    bytes = 0;
  }
  void ensure(size_t need)
  {
    if (need <= bytes && p) return;
    release();
    const size_t want = std::max<size_t>(need + need / 8, 4096);
    if (hipHostMalloc(&p, want, hipHostMallocDefault) != hipSuccess) {
      p = nullptr;
      (void) hipGetLastError();
      throw std::bad_alloc();
    }
    bytes = want;
  }
  template<class U> U *as() const { return static_cast<U *>(p); }
};

template<class U> void upload_vec(DevBuf &b, const std::vector<U> &v)
{
  b.ensure(std::max<size_t>(v.size(), 1) * sizeof(U));
  if (!v.empty()) HIP_CHECK(hipMemcpy(b.p, v.data(), v.size() * sizeof(U), hipMemcpyHostToDevice));
}

inline int round_up(int a, int b) { return (a + b - 1) / b * b; }

struct HostProd {
  std::vector<int> off, l, r;
  std::vector<double> c;
  std::vector<int> loff, l_o, l_r, roff, r_o, r_l;
  std::vector<double> l_c, r_c;
  std::vector<ProdTerm> terms;    // the kept terms, for the specialised kernels
  int nout = 0, nleft = 0, nright = 0;
};

// terms of outputs with need[o] set, sorted by output; operand-major copies for the reverse
inline HostProd build_prod(const CGProduct &p, const std::vector<char> &need, int nleft, int nright)
{
  HostProd h;
  h.nout = p.n_out;
  h.nleft = nleft;
  h.nright = nright;
  std::vector<int> ord;
  for (int t = 0; t < p.n_terms; t++)
    if (need[p.m_sum_ind[t]]) ord.push_back(t);
  std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return p.m_sum_ind[a] < p.m_sum_ind[b]; });
  h.off.assign(h.nout + 1, 0);
  for (int t : ord) {
    h.l.push_back(p.left_ind[t]);
    h.r.push_back(p.right_ind[t]);
    h.c.push_back(p.cg_coeff[t]);
    h.off[p.m_sum_ind[t] + 1]++;
    h.terms.push_back({p.left_ind[t], p.right_ind[t], p.m_sum_ind[t], p.cg_coeff[t]});
  }
  for (int o = 0; o < h.nout; o++) h.off[o + 1] += h.off[o];
  auto by_operand = [&](const std::vector<int> &key, int nkey, std::vector<int> &off, std::vector<int> &oo,
                        std::vector<int> &other, std::vector<double> &cc, const std::vector<int> &oth) {
    std::vector<int> o2 = ord;
    std::stable_sort(o2.begin(), o2.end(), [&](int a, int b) { return key[a] < key[b]; });
    off.assign(nkey + 1, 0);
    for (int t : o2) {
      oo.push_back(p.m_sum_ind[t]);
      other.push_back(oth[t]);
      cc.push_back(p.cg_coeff[t]);
      off[key[t] + 1]++;
    }
    for (int q = 0; q < nkey; q++) off[q + 1] += off[q];
  };
  by_operand(p.left_ind, nleft, h.loff, h.l_o, h.l_r, h.l_c, p.right_ind);
  by_operand(p.right_ind, nright, h.roff, h.r_o, h.r_l, h.r_c, p.left_ind);
  return h;
}

struct DevProd {
  DevBuf off, l, r, c, loff, l_o, l_r, l_c, roff, r_o, r_l, r_c;
  ProdDev d{};
  JitKernels jit;        // model-specialised kernels (jit_prod.hpp); not ok(): the table-driven kernels run
  std::string jit_note;
  ~DevProd() { jit.release(); }
  void build(const HostProd &h)
  {
    upload_vec(off, h.off); upload_vec(l, h.l); upload_vec(r, h.r); upload_vec(c, h.c);
    upload_vec(loff, h.loff); upload_vec(l_o, h.l_o); upload_vec(l_r, h.l_r); upload_vec(l_c, h.l_c);
    upload_vec(roff, h.roff); upload_vec(r_o, h.r_o); upload_vec(r_l, h.r_l); upload_vec(r_c, h.r_c);
    d.off = off.as<int>(); d.l = l.as<int>(); d.r = r.as<int>(); d.c = c.as<double>();
    d.loff = loff.as<int>(); d.l_o = l_o.as<int>(); d.l_r = l_r.as<int>(); d.l_c = l_c.as<double>();
    d.roff = roff.as<int>(); d.r_o = r_o.as<int>(); d.r_l = r_l.as<int>(); d.r_c = r_c.as<double>();
    d.nout = h.nout; d.nleft = h.nleft; d.nright = h.nright;
  }
};

// weights W[K][N] (row-major) of a tile GEMM in MFMA fragment order [cb][s][lane]: lane (g, c) holds
// W[g * (K / 4) + s][cb * 16 + c]
// (k index frag_k<T>, or g * Kp / 4 + s with plain: inputs that are no rows of a multiple of 16 channels)
template<class T> void pack_fragments(const std::vector<double> &W, int K, int N, int Kp, int Np, std::vector<T> &out, bool plain = false)
{
  const int ks = Kp / 4, nb = Np / 16;
  const size_t base = out.size();
  out.resize(base + (size_t) nb * ks * 64, (T) 0);
  for (int cb = 0; cb < nb; cb++)
    for (int s = 0; s < ks; s++)
      for (int lane = 0; lane < 64; lane++) {
        const int g = lane >> 4, c = lane & 15, k = plain ? g * ks + s : frag_k<T>(g, s), n = cb * 16 + c;
        if (k < K && n < N) out[base + ((size_t) cb * ks + s) * 64 + lane] = (T) W[(size_t) k * N + n];
      }
}

template<class T> struct DevJobs {
  DevBuf job_out, job_scale, job_dst, job_add, seg_off, seg_src, seg_fn, seg_w, seg_scale, seg;
  GemmJobs<T> d{};
  long long nseg[2] = {0, 0};    // segments that read source 0 / source 1
  long long seg_count = 0;
  struct Host {
    std::vector<int> job_out, job_dst, seg_off{0}, seg_src, seg_fn, seg_w;
    std::vector<T> job_scale, job_add, seg_scale;     // job_add: empty, or a factor for every job
    void job(int out, double scale, int dst = 0) { job_out.push_back(out); job_scale.push_back((T) scale); job_dst.push_back(dst); }
    void seg(int src, int fn, int w, double scale) { seg_src.push_back(src); seg_fn.push_back(fn); seg_w.push_back(w); seg_scale.push_back((T) scale); }
    void end_job() { seg_off.push_back((int) seg_src.size()); }
  };
  void build(const Host &h, const T *WF0, const T *WF1)
  {
    upload_vec(job_out, h.job_out); upload_vec(job_scale, h.job_scale); upload_vec(seg_off, h.seg_off);
    upload_vec(seg_src, h.seg_src); upload_vec(seg_fn, h.seg_fn); upload_vec(seg_w, h.seg_w); upload_vec(seg_scale, h.seg_scale);
    d.job_out = job_out.as<int>(); d.job_scale = job_scale.as<T>(); d.seg_off = seg_off.as<int>();
    d.seg_src = seg_src.as<int>(); d.seg_fn = seg_fn.as<int>(); d.seg_w = seg_w.as<int>(); d.seg_scale = seg_scale.as<T>();
    upload_vec(job_dst, h.job_dst);
    if (!h.job_add.empty()) upload_vec(job_add, h.job_add);
    std::vector<int4> sv;
    for (size_t q = 0; q < h.seg_src.size(); q++) sv.push_back(int4{h.seg_src[q], h.seg_fn[q], h.seg_w[q], 0});
    if (sv.empty()) sv.push_back(int4{0, 0, 0, 0});
    upload_vec(seg, sv);
    d.job_dst = job_dst.as<int>(); d.seg = seg.as<int4>(); d.job_add = h.job_add.empty() ? nullptr : job_add.as<T>();
    d.WF0 = WF0; d.WF1 = WF1;
    d.njobs = (int) h.job_out.size();
    nseg[0] = nseg[1] = 0;
    seg_count = (long long) h.seg_src.size();
    for (int src : h.seg_src) nseg[src ? 1 : 0]++;
    d.max_seg = 0;
    for (size_t q = 0; q + 1 < h.seg_off.size(); q++) d.max_seg = std::max(d.max_seg, h.seg_off[q + 1] - h.seg_off[q]);
  }
  void set_rows(const int *drow) { for (int q = 0; q < 16; q++) d.drow[q] = drow[q]; }
};

// One FC layer as three job lists (forward, reverse into the left input, reverse into the right input) over
// fragment-ordered weight tiles.  Widths are the padded ones (multiples of 16; padding weights are zero).
template<class T> struct DevFc {
  DevBuf WlF, WrF, WlTF, WrTF;
  DevJobs<T> fwd, bwd_l, bwd_r;
  // the reverse of a layer whose two inputs are ONE tensor (A1 = FC(A, A)): a job per input function that takes the left
  // segment and the right segments together (source 0: left weights, source 1: right weights; both sources are the output
  // adjoint), one launch and one read-add-write of the input adjoint instead of two; empty unless build() was asked for it
  DevJobs<T> bwd_lr;
  bool have_lr = false;
  int nil = 0, nir = 0, no = 0;    // padded widths
  // nfr: functions of the right-input tensor; livef: outputs that are computed; cover_left: the reverse into the left
  // input has a job for EVERY function (without segments for outputs that are not computed), so that a launch that
  // overwrites instead of accumulating leaves no row of the adjoint unwritten
  void build(const FCWeights &w, const std::vector<char> &livef, int nfr, int nil_p, int nir_p, int no_p, const int *drow,
             bool cover_left = false, bool same_input = false)
  {
    nil = nil_p; nir = nir_p; no = no_p;
    const int nt = w.tiles_left;
    std::vector<T> fl, fr, flt, frt;
    std::vector<double> M, Mt;
    auto tile_mats = [&](const std::vector<double> &W, double norm, int nin, int t) {
      M.assign((size_t) nin * w.n_out, 0.0);     // [n][k]
      Mt.assign((size_t) w.n_out * nin, 0.0);    // [k][n]
      for (int k = 0; k < w.n_out; k++)
        for (int n = 0; n < nin; n++) {
          const double v = norm * W[((size_t) k * nin + n) * nt + t];
          M[(size_t) n * w.n_out + k] = v;
          Mt[(size_t) k * nin + n] = v;
        }
    };
    for (int t = 0; t < nt; t++) {
      tile_mats(w.w_left, w.norm_left, w.n_in_left, t);
      pack_fragments<T>(M, w.n_in_left, w.n_out, nil, no, fl);
      pack_fragments<T>(Mt, w.n_out, w.n_in_left, no, nil, flt);
      tile_mats(w.w_right, w.norm_right, w.n_in_right, t);
      pack_fragments<T>(M, w.n_in_right, w.n_out, nir, no, fr);
      pack_fragments<T>(Mt, w.n_out, w.n_in_right, no, nir, frt);
    }
    upload_vec(WlF, fl); upload_vec(WrF, fr); upload_vec(WlTF, flt); upload_vec(WrTF, frt);
    typename DevJobs<T>::Host hf, hl, hr;
    std::vector<std::vector<int>> conn_of(w.n_funcs), conn_from(nfr);
    for (int c = 0; c < w.n_conn; c++) {
      conn_of[w.collect_to[c]].push_back(c);
      if (livef[w.collect_to[c]]) conn_from[w.collect_from[c]].push_back(c);
    }
    for (int f = 0; f < w.n_funcs; f++) {
      if (!livef[f]) {
        if (cover_left) { hl.job(f, 1.0); hl.end_job(); }
        continue;
      }
      hf.job(f, w.norm_out_factor[f]);
      hf.seg(0, f, w.w_tile_left[f], 1.0);
      for (int c : conn_of[f]) hf.seg(1, w.collect_from[c], w.w_tile_right[c], 1.0);
      hf.end_job();
      hl.job(f, w.norm_out_factor[f]);
      hl.seg(0, f, w.w_tile_left[f], 1.0);
      hl.end_job();
    }
    for (int r = 0; r < nfr; r++) {
      if (conn_from[r].empty()) continue;
      hr.job(r, 1.0);
      for (int c : conn_from[r]) hr.seg(0, w.collect_to[c], w.w_tile_right[c], w.norm_out_factor[w.collect_to[c]]);
      hr.end_job();
    }
    fwd.build(hf, WlF.as<T>(), WrF.as<T>());
    bwd_l.build(hl, WlTF.as<T>(), WlTF.as<T>());
    bwd_r.build(hr, WrTF.as<T>(), WrTF.as<T>());
    fwd.set_rows(drow); bwd_l.set_rows(drow); bwd_r.set_rows(drow);
    have_lr = same_input && nil == nir && nfr == w.n_funcs;
    if (have_lr) {
      typename DevJobs<T>::Host hlr;
      for (int r = 0; r < nfr; r++) {
        if (!livef[r] && conn_from[r].empty()) continue;
        hlr.job(r, 1.0);
        if (livef[r]) hlr.seg(0, r, w.w_tile_left[r], w.norm_out_factor[r]);
        for (int c : conn_from[r]) hlr.seg(1, w.collect_to[c], w.w_tile_right[c], w.norm_out_factor[w.collect_to[c]]);
        hlr.end_job();
      }
      bwd_lr.build(hlr, WlTF.as<T>(), WrTF.as<T>());
      bwd_lr.set_rows(drow);
    }
  }
};

// The reverse of two FC layers that read the same two inputs (AA1 = FC1(AA, A), AA2 = FC2(AA, A)) as ONE pair of job
// lists: the adjoint of the shared left input is read, added to and written once instead of twice, and so is the
// adjoint of the right input.  Source 0 of a segment is the output adjoint of the first layer, source 1 of the second.
template<class T> struct DevFcPairBwd {
  DevJobs<T> bwd_l, bwd_r;
  // cover_left: the reverse into the left input has a job for EVERY function (those no live output reads get one without
  // segments), so that a launch that overwrites instead of accumulating leaves no row of the adjoint unwritten
  void build(const FCWeights &w1, const std::vector<char> &live1, const DevFc<T> &F1, const FCWeights &w2, const std::vector<char> &live2,
             const DevFc<T> &F2, int nfr, const int *drow, bool cover_left = false)
  {
    if (w1.n_funcs != w2.n_funcs || F1.nil != F2.nil || F1.nir != F2.nir || F1.no != F2.no) throw Error("FC pair: the two layers differ in shape");
    typename DevJobs<T>::Host hl, hr;
    for (int f = 0; f < w1.n_funcs; f++) {
      if (!live1[f] && !live2[f] && !cover_left) continue;
      hl.job(f, 1.0);
      if (live1[f]) hl.seg(0, f, w1.w_tile_left[f], w1.norm_out_factor[f]);
      if (live2[f]) hl.seg(1, f, w2.w_tile_left[f], w2.norm_out_factor[f]);
      hl.end_job();
    }
    std::vector<std::vector<std::pair<int, int>>> from(nfr);    // (layer, connection)
    for (int c = 0; c < w1.n_conn; c++)
      if (live1[w1.collect_to[c]]) from[w1.collect_from[c]].push_back({0, c});
    for (int c = 0; c < w2.n_conn; c++)
      if (live2[w2.collect_to[c]]) from[w2.collect_from[c]].push_back({1, c});
    for (int r = 0; r < nfr; r++) {
      if (from[r].empty()) continue;
      hr.job(r, 1.0);
      for (const auto &lc : from[r]) {
        const FCWeights &w = lc.first ? w2 : w1;
        const int c = lc.second;
        hr.seg(lc.first, w.collect_to[c], w.w_tile_right[c], w.norm_out_factor[w.collect_to[c]]);
      }
      hr.end_job();
    }
    bwd_l.build(hl, F1.WlTF.template as<T>(), F2.WlTF.template as<T>());
    bwd_r.build(hr, F1.WrTF.template as<T>(), F2.WrTF.template as<T>());
    bwd_l.set_rows(drow); bwd_r.set_rows(drow);
  }
};


// The bonds of a pass whose radial rows are evaluated (k_edge_pairs): uid / x [*n], erow [bonds]; on == false: every bond has
// its own row
struct PairedRows {
  bool on = false;
  const int *uid = nullptr, *erow = nullptr;
  const double *x = nullptr;
  const long long *n = nullptr;
};

// A 3-layer radial MLP in MFMA fragment order and the launch of the persistent radial kernel (radial_x.h:11-60 of the
// reference; its spline tables are replaced by the exact network).  Output column l * CP + n of an edge holds
// R_{n,l}(x) z[mu_j][n] (file order of the last layer: o = n nl + l, libgrace/src/fused_1l.cpp:123).
template<class T> struct DevRadial {
  DevBuf w0, w1, w2, bias_i, bias_j, bias1;
  // radial tables (the reference's spline_n, libgrace/include/grace/system.h:78): intervals asked for (0: the MLP itself is
  // evaluated for every bond) and the table that exists: value and d/dx at the knots, [N + 1][noutp] each
  int spline_n = 0, table_n = 0;
  DevBuf tabF, tabD, knots, knot_mu, knot_mi, unit_z, knotF, knotD;
  // species form: the species of the engine (elements that atom types map to), element -> species, and the memory the pair
  // tables may take (the reference's spline_mb, libgrace/include/grace/system.h:85: beyond it the MLP itself is evaluated)
  std::vector<int> species_mu;
  DevBuf sp_of_mu;
  bool tables_allowed = true;
  std::string who_tables = "radial tables";
  void set_species(const std::vector<int> &present_mu, int n_elements, const std::string &who)
  {
    species_mu = present_mu;
    std::vector<int> map((size_t) n_elements, 0);
    for (size_t q = 0; q < species_mu.size(); q++) map[(size_t) species_mu[q]] = (int) q;
    upload_vec(sp_of_mu, map);
    who_tables = who;
  }
  // bytes of the tables of `n` intervals for the engine's species pairs
  double table_bytes(int n) const
  {
    const double pairs = mode == 1 ? (double) species_mu.size() * species_mu.size() : 1.0;
    return sizeof(T) == 8 ? pairs * (n + 1.0) * noutp * 16.0 : pairs * n * 4.0 * noutp * 4.0;
  }
  // fp32 engines: the same MLP in fp64, which evaluates the knots of the tables (build_double)
  std::unique_ptr<DevRadial<double>> dbl;
  template<class... A> void build_double(A &&...a)
  {
    if constexpr (sizeof(T) == 4) {
      dbl = std::make_unique<DevRadial<double>>();
      dbl->build(std::forward<A>(a)...);
    }
  }
  template<class... A> void build_species_double(A &&...a)
  {
    if constexpr (sizeof(T) == 4) {
      dbl = std::make_unique<DevRadial<double>>();
      dbl->build_species(std::forward<A>(a)...);
    }
  }
  int mode = 0;    // 1: species form (build_species)
  int hb = 4, ks0 = 2, nob = 0, noutp = 0, w2_in_lds = 1, nrb = 0, p = 0, act = 0, CP = 0, nel = 0;
  size_t lds = 0;
  int drow[16];
  void build(const std::vector<MLPLayer> &mlp, int nradbase, int basis_p, int activation, int C, int CP_, int nl, int nel_,
             const int *drow_, const std::string &who)
  {
    if (mlp.size() != 3)
      throw Error(who + ": the GPU radial kernel implements 3-layer radial MLPs (file has " + std::to_string(mlp.size()) + ")");
    const MLPLayer &L0 = mlp[0], &L1 = mlp[1], &L2 = mlp[2];
    const int H1 = L0.n_out, H2 = L1.n_out;
    if (nradbase > kMaxRadBasis) throw Error(who + ": nradbase > 16 not supported");
    const int hmax = std::max(H1, H2);
    if (hmax <= 64) hb = 4;
    else if (hmax <= 128) hb = 8;
    else throw Error(who + ": radial MLP hidden width > 128 not supported");
    nrb = nradbase; p = basis_p; act = activation; CP = CP_; nel = nel_;
    for (int q = 0; q < 16; q++) drow[q] = drow_[q];
    ks0 = round_up(nradbase, 4) / 4;
    const int nout = CP * nl;
    noutp = round_up(nout, 16);
    nob = noutp / 16;
    std::vector<T> v0((size_t) hb * ks0 * 64, (T) 0), v1((size_t) hb * hb * 4 * 64, (T) 0), v2(((size_t) nob * hb * 4 + kRadialPrefetch) * 64, (T) 0);
    for (int rb = 0; rb < hb; rb++)
      for (int s = 0; s < ks0; s++)
        for (int lane = 0; lane < 64; lane++) {
          const int g = lane >> 4, r = lane & 15, kin = 4 * s + g, out = rb * 16 + r;
          if (kin < L0.n_in && out < H1) v0[((size_t) rb * ks0 + s) * 64 + lane] = (T) (L0.norm * L0.W[(size_t) kin * H1 + out]);
        }
    for (int rb = 0; rb < hb; rb++)
      for (int kb = 0; kb < hb; kb++)
        for (int s = 0; s < 4; s++)
          for (int lane = 0; lane < 64; lane++) {
            const int g = lane >> 4, r = lane & 15, in = kb * 16 + drow[g * 4 + s], out = rb * 16 + r;
            if (in < H1 && out < H2) v1[(((size_t) rb * hb + kb) * 4 + s) * 64 + lane] = (T) (L1.norm * L1.W[(size_t) in * H2 + out]);
          }
    for (int cb = 0; cb < nob; cb++)
      for (int kb = 0; kb < hb; kb++)
        for (int s = 0; s < 4; s++)
          for (int lane = 0; lane < 64; lane++) {
            const int g = lane >> 4, cc = lane & 15, in = kb * 16 + drow[g * 4 + s], col = cb * 16 + cc;
            const int l = col / CP, n = col % CP, o = n * nl + l;
            if (in < H2 && col < nout && n < C)
              v2[(((size_t) cb * hb + kb) * 4 + s) * 64 + lane] = (T) (L2.norm * L2.W[(size_t) in * L2.n_out + o]);
          }
    upload_vec(w0, v0); upload_vec(w1, v1); upload_vec(w2, v2);
    const size_t base = (v0.size() + v1.size()) * sizeof(T);
    w2_in_lds = base + v2.size() * sizeof(T) <= 150 * 1024;
    lds = base + (w2_in_lds ? v2.size() * sizeof(T) : 0);
  }
  // Species form of GRACE-3L (libgrace/src/fused_3l.cpp:299-346, :462-493): the MLP input is [T_1..T_nrb(2x - 1),
  // emb(mu_i), emb(mu_j)], hidden layers carry a bias, and the envelope multiplies the output.  The embedding rows of
  // layer 0 become per-element tables added to its pre-activation: tab_i[mu] = norm0 (b0 + emb[mu] W0[nrb : nrb + ne]),
  // tab_j[mu] = norm0 emb[mu] W0[nrb + ne : nrb + 2 ne].
  void build_species(const std::vector<MLPLayer> &mlp, const std::vector<std::vector<double>> &bias, const std::vector<double> &emb, int ne,
                     int nradbase, int basis_p, int C, int CP_, int nl, int nel_, const int *drow_, const std::string &who)
  {
    if (mlp.size() != 3)
      throw Error(who + ": the GPU radial kernel implements 3-layer radial MLPs (file has " + std::to_string(mlp.size()) + ")");
    std::vector<MLPLayer> cut = mlp;
    const int H1 = mlp[0].n_out, H2 = mlp[1].n_out;
    cut[0].n_in = nradbase;
    cut[0].W.assign(mlp[0].W.begin(), mlp[0].W.begin() + (size_t) nradbase * H1);
    build(cut, nradbase, basis_p, 0, C, CP_, nl, nel_, drow_, who);
    mode = 1;
    const int HP = hb * 16;
    std::vector<T> ti((size_t) nel_ * HP, (T) 0), tj((size_t) nel_ * HP, (T) 0), t1((size_t) HP, (T) 0);
    for (int mu = 0; mu < nel_; mu++)
      for (int o = 0; o < H1; o++) {
        double vi = bias.size() > 0 && !bias[0].empty() ? bias[0][o] : 0.0, vj = 0.0;
        for (int e = 0; e < ne; e++) {
          const double zz = emb[(size_t) mu * ne + e];
          vi += zz * mlp[0].W[(size_t) (nradbase + e) * H1 + o];
          vj += zz * mlp[0].W[(size_t) (nradbase + ne + e) * H1 + o];
        }
        ti[(size_t) mu * HP + o] = (T) (mlp[0].norm * vi);
        tj[(size_t) mu * HP + o] = (T) (mlp[0].norm * vj);
      }
    for (int o = 0; o < H2; o++) t1[o] = (T) (bias.size() > 1 && !bias[1].empty() ? mlp[1].norm * bias[1][o] : 0.0);
    if (bias.size() > 2 && !bias[2].empty()) throw Error(who + ": a bias on the output layer of the radial MLP is not supported");
    upload_vec(bias_i, ti); upload_vec(bias_j, tj); upload_vec(bias1, t1);
  }
  // z: [nel][CP] species weights of the neighbour (null, only where tables are used: rows without weights); e_count < 0: the
  // edge count is read from *n_edges on the device; emi: element of the central atom of every edge (species form only)
  // tables: use the radial tables when the engine was asked for them (the plain form only); otherwise, and for the debug
  // entry points, the MLP is evaluated for every bond.  listed: no more edges than this where e_count < 0 (< 0: not known)
  void launch(hipStream_t stream, int ncu, const T *z, long long e_begin, long long e_count, const double *x, const int *emu, T *Rz, T *dRz,
              const long long *n_edges, const int *emi = nullptr, bool tables = false, long long listed = -1)
  {
    if (tables && has_tables()) {
      ensure_tables(stream, ncu);
      const long long bound = e_count >= 0 ? e_count : (long long) 1 << 40;
      const unsigned grid = (unsigned) std::max<long long>(1, std::min<long long>(bound, (long long) ncu * 32));
      auto kern = z ? k_radial_spline<T, sizeof(T) == 4, true> : k_radial_spline<T, sizeof(T) == 4, false>;
      hipLaunchKernelGGL(kern, dim3(grid), dim3(round_up(noutp, 64)), 0, stream, n_edges, e_begin, e_count, x, emu,
                         (const T *) tabF.template as<T>(), (const T *) tabD.template as<T>(), table_n, z, CP, noutp, Rz, dRz,
                         mode == 1 ? emi : (const int *) nullptr, (const int *) sp_of_mu.as<int>(), (int) species_mu.size());
      return;
    }
    launch_mlp(stream, ncu, z, e_begin, e_count, x, emu, Rz, dRz, n_edges, emi, listed);
  }
  // only the listed rows, without the species weights (the plain form; no tables)
  void launch_paired(hipStream_t stream, int ncu, const PairedRows &rows, T *Rz, T *dRz)
  {
    RadialArgs<T> ra = mlp_args(nullptr, 0, -1, rows.x, nullptr, Rz, dRz, rows.n, nullptr);
    ra.uid = rows.uid;
    run_mlp<true>(stream, ncu, ra, -1);
  }
  // tables requested (spline_n > 0) and, in the species form, within the memory they may take
  bool has_tables()
  {
    if (spline_n <= 0) return false;
    if (mode == 0) return true;
    if (species_mu.empty()) return false;
    return tables_allowed;
  }
  // the tables as the kernels that evaluate them take them (built on first use and again after release_buffers)
  RadialTable<T> table(hipStream_t stream, int ncu, const double *x, const int *emu, const T *z)
  {
    ensure_tables(stream, ncu);
    RadialTable<T> t{};
    t.F = tabF.template as<T>();
    t.D = tabD.template as<T>();
    t.N = table_n;
    t.x = x;
    t.emu = emu;
    t.z = z;
    return t;
  }
  void ensure_tables(hipStream_t stream, int ncu)
  {
    {
      const int N = spline_n;
      if (table_n != N || !tabF.p || (sizeof(T) == 8 && !tabD.p)) {    // the MLP at the knots x = k / N, unit species weights (again after release_buffers)
        // species form: the knots of every ordered pair of species, pair after pair
        const size_t nsp = mode == 1 ? species_mu.size() : 1, npair = nsp * nsp;
        std::vector<double> xs(((size_t) N + 1) * npair);
        std::vector<int> kmi(xs.size(), 0), kmj(xs.size(), 0);
        for (size_t pr = 0; pr < npair; pr++)
          for (int k = 0; k <= N; k++) {
            const size_t q = pr * ((size_t) N + 1) + k;
            xs[q] = (double) k / N;
            if (mode == 1) { kmi[q] = species_mu[pr / nsp]; kmj[q] = species_mu[pr % nsp]; }
          }
        upload_vec(knots, xs);
        upload_vec(knot_mu, kmj);
        upload_vec(knot_mi, kmi);
        const long long nknots = (long long) xs.size();
        const size_t rows = xs.size() * noutp;
        if constexpr (sizeof(T) == 8) {
          upload_vec(unit_z, std::vector<T>((size_t) CP * std::max(nel, 1), (T) 1));
          tabF.ensure(rows * sizeof(T));
          tabD.ensure(rows * sizeof(T));
          launch_mlp(stream, ncu, unit_z.template as<T>(), 0, nknots, knots.as<double>(), knot_mu.as<int>(), tabF.template as<T>(),
                     tabD.template as<T>(), nullptr, mode == 1 ? knot_mi.as<int>() : nullptr);
        } else {
          if (!dbl) throw Error("radial tables of an fp32 engine need the fp64 form of its radial MLP");
          upload_vec(unit_z, std::vector<double>((size_t) CP * std::max(nel, 1), 1.0));
          knotF.ensure(rows * sizeof(double));
          knotD.ensure(rows * sizeof(double));
          tabF.ensure(npair * (size_t) N * 4 * noutp * sizeof(T));
          dbl->launch_mlp(stream, ncu, unit_z.as<double>(), 0, nknots, knots.as<double>(), knot_mu.as<int>(), knotF.as<double>(),
                          knotD.as<double>(), nullptr, mode == 1 ? knot_mi.as<int>() : nullptr);
          const long long tot = (long long) N * noutp;
          for (size_t pr = 0; pr < npair; pr++)
            hipLaunchKernelGGL(k_spline_coef, dim3((unsigned) ((tot + 255) / 256)), dim3(256), 0, stream,
                               (const double *) knotF.as<double>() + pr * ((size_t) N + 1) * noutp,
                               (const double *) knotD.as<double>() + pr * ((size_t) N + 1) * noutp, N, noutp,
                               tabF.as<float>() + pr * (size_t) N * 4 * noutp);
          knotF.release();    // the fp64 knots are needed for the coefficients only
          knotD.release();
        }
        table_n = N;
      }
    }
  }
  // the radial MLP itself for every edge of the range
  void launch_mlp(hipStream_t stream, int ncu, const T *z, long long e_begin, long long e_count, const double *x, const int *emu, T *Rz, T *dRz,
                  const long long *n_edges, const int *emi, long long listed = -1)
  {
    if (mode == 1 && !emi) throw Error("radial kernel: the species form needs the central element of every edge");
    run_mlp<false>(stream, ncu, mlp_args(z, e_begin, e_count, x, emu, Rz, dRz, n_edges, emi), e_count >= 0 ? e_count : listed);
  }
  RadialArgs<T> mlp_args(const T *z, long long e_begin, long long e_count, const double *x, const int *emu, T *Rz, T *dRz, const long long *n_edges,
                         const int *emi) const
  {
    RadialArgs<T> ra{};
    ra.n_edges = n_edges;
    ra.e_begin = e_begin;
    ra.e_count = e_count;
    ra.x = x;
    ra.emu = emu;
    ra.w0 = w0.as<T>(); ra.w1 = w1.as<T>(); ra.w2 = w2.as<T>();
    ra.z = z;
    ra.Rz = Rz; ra.dRz = dRz;
    ra.nrb = nrb; ra.p = p; ra.ks0 = ks0;
    ra.nob = nob; ra.noutp = noutp;
    ra.C = CP; ra.nel = nel; ra.act = act;
    ra.w2_in_lds = w2_in_lds;
    for (int q = 0; q < 16; q++) ra.drow[q] = drow[q];
    ra.emi = emi; ra.bias_i = bias_i.as<T>(); ra.bias_j = bias_j.as<T>(); ra.bias1 = bias1.as<T>();
    return ra;
  }
  // <T, 16-row blocks of the hidden width, activation, species form, layer-2 weights in LDS, listed rows>
  template<bool W2L, bool LISTED> auto mlp_kernel() const
  {
    auto kern = hb == 4 ? (act == 1 ? k_radial<T, 4, 1, 0, W2L, LISTED> : k_radial<T, 4, 0, 0, W2L, LISTED>)
                        : (act == 1 ? k_radial<T, 8, 1, 0, W2L, LISTED> : k_radial<T, 8, 0, 0, W2L, LISTED>);
    if constexpr (!LISTED) if (mode == 1) kern = hb == 4 ? k_radial<T, 4, 0, 1, W2L, false> : k_radial<T, 8, 0, 1, W2L, false>;
    return kern;
  }
  // most: no more edges than this (< 0: not known).  Up to three tiles of 16 edges per CU at width 64 and two at width 128 the
  // waves of a block share a tile (times at k_radial_few).
  template<bool LISTED> void run_mlp(hipStream_t stream, int ncu, const RadialArgs<T> &ra, long long most)
  {
    const long long tiles = (most + 15) / 16;
    if (!LISTED && most > 0 && tiles <= (hb == 4 ? 3 : 2) * (long long) ncu) {
      auto few = mode == 1 ? (hb == 4 ? k_radial_few<T, 4, 0, 1> : k_radial_few<T, 8, 0, 1>)
               : hb == 4   ? (act == 1 ? k_radial_few<T, 4, 1, 0> : k_radial_few<T, 4, 0, 0>)
                           : (act == 1 ? k_radial_few<T, 8, 1, 0> : k_radial_few<T, 8, 0, 0>);
      const size_t bytes = (size_t) radial_few_lds(hb) * sizeof(T);
      if (bytes > 48 * 1024) HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(few), hipFuncAttributeMaxDynamicSharedMemorySize, (int) bytes));
      hipLaunchKernelGGL(few, dim3((unsigned) tiles), dim3(64 * hb), bytes, stream, ra);
      return;
    }
    const int threads = radial_threads(hb, mode, w2_in_lds != 0);
    auto kern = w2_in_lds ? mlp_kernel<true, LISTED>() : mlp_kernel<false, LISTED>();
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    hipLaunchKernelGGL(kern, dim3(ncu), dim3(threads), lds, stream, ra);
  }
};

// One source of an element-dependent reduce, as the host containers give it (weights [nel][nout][nin][w_shape])
struct ReduceSrc {
  const std::vector<double> *W;
  double norm;
  int n_in, w_shape;
  const std::vector<int> *collect_ind, *w_l_tile, *out_fn;    // out_fn: output function per connection, or null (one function)
  int nfun, ninp;                                            // functions of the source tensor, its padded channel width
};

// functions of source w that the reduce collects (fo >= 0: through the connections whose output function is fo)
inline std::vector<int> reduce_functions(const ReduceSrc &w, int fo)
{
  std::vector<int> fn;
  for (size_t c = 0; c < w.collect_ind->size(); c++)
    if (fo < 0 || !w.out_fn || (*w.out_fn)[c] == fo) fn.push_back((*w.collect_ind)[c]);
  std::sort(fn.begin(), fn.end());
  fn.erase(std::unique(fn.begin(), fn.end()), fn.end());
  return fn;
}
// M[n][k] of function fn for element mu: the sum of its connections' weight tiles
inline void reduce_matrix(const ReduceSrc &w, int fo, int fn, int mu, int nout, std::vector<double> &M)
{
  const int nin = w.n_in;
  M.assign((size_t) nin * nout, 0.0);
  for (size_t c = 0; c < w.collect_ind->size(); c++) {
    if ((*w.collect_ind)[c] != fn || (fo >= 0 && w.out_fn && (*w.out_fn)[c] != fo)) continue;
    const int tile = (*w.w_l_tile)[c];
    for (int k = 0; k < nout; k++)
      for (int n = 0; n < nin; n++) M[(size_t) n * nout + k] += w.norm * (*w.W)[(((size_t) mu * nout + k) * nin + n) * w.w_shape + tile];
  }
}

// One element-dependent reduce of a set: up to 4 sources into `nout` channels of ONE output function
// (fused_cpu.h:1202-1273 of the reference).  fo >= 0 keeps the connections whose output function is fo.  sel: array of the
// result (0: fp64 rows, 1: rows of the engine's type), ostride / ooff: its row in that array.
struct ReduceSpec {
  std::vector<ReduceSrc> src;
  int nout = 0, fo = -1, sel = 0, ostride = 0, ooff = 0;
};

// Reduces that read the same tensors: one launch forward, one launch in the reverse, where every adjoint row is visited once
// whatever number of reduces feed it (k_reduce_fwd, k_reduce_bwd).
template<class T> struct DevReduces {
  std::vector<std::unique_ptr<DevBuf>> bufs;
  std::vector<ReduceDev<T>> d;
  int max_jobs = 0;    // collected functions of the longest reduce
  // reverse: rows of the sources s >= 2, and of s < 2, and all of them.  A list is a sequence of launches (rows fed by more
  // than two reduces take a second one, which adds)
  struct List {
    std::vector<ReduceBwdJob> host;
    DevBuf dev;
  };
  std::vector<std::unique_ptr<List>> high, low, all;
  DevBuf WB;
  RowMap drow{};

  // cover: functions of source 0 whose adjoint row the list `all` writes although no reduce collects them
  void build(const std::vector<ReduceSpec> &specs, int nel, const int *drow_, const std::vector<char> &cover = {})
  {
    for (int q = 0; q < 16; q++) drow.r[q] = drow_[q];
    const int ns = specs.empty() ? 0 : (int) specs[0].src.size();
    std::map<std::pair<int, int>, std::vector<int>> fed;    // (source, function) -> the reduces that collect it
    std::vector<double> M, Mt;
    for (size_t r = 0; r < specs.size(); r++) {
      const ReduceSpec &sp = specs[r];
      if (sp.nout > 32) throw Error("reduce widths above 32 are not supported by the GPU reduce kernels");
      ReduceDev<T> x{};
      x.nsrc = ns;
      x.nrho = sp.nout;
      x.nbr = (sp.nout + 15) / 16;
      x.sel = sp.sel;
      x.ostride = sp.ostride;
      x.ooff = sp.ooff;
      for (int q = 0; q < 16; q++) x.drow[q] = drow_[q];
      int jobs = 0;
      for (int s = 0; s < ns; s++) {
        const ReduceSrc &w = sp.src[s];
        const std::vector<int> fn = reduce_functions(w, sp.fo);
        std::vector<T> vF;
        for (int mu = 0; mu < nel; mu++)
          for (int f : fn) {
            reduce_matrix(w, sp.fo, f, mu, sp.nout, M);
            pack_fragments<T>(M, w.n_in, sp.nout, w.ninp, x.nbr * 16, vF);    // X[atom][n] . M[n][k]
          }
        for (int f : fn) fed[{s, f}].push_back((int) r);
        bufs.emplace_back(new DevBuf());
        upload_vec(*bufs.back(), vF);
        x.WF[s] = bufs.back()->template as<T>();
        bufs.emplace_back(new DevBuf());
        upload_vec(*bufs.back(), fn);
        x.fn[s] = bufs.back()->template as<int>();
        x.ncol[s] = (int) fn.size();
        x.nin[s] = w.ninp;
        x.stride[s] = w.nfun;
        jobs += (int) fn.size();
      }
      max_jobs = std::max(max_jobs, jobs);
      d.push_back(x);
    }
    // reverse: g[atom][k] . W[k][n], weights [job][mu][con][cb < 2][step < 8][lane]
    std::vector<T> vB;
    auto add_rows = [&](int s, int f, const std::vector<int> &reds) {
      const ReduceSrc &w0 = specs[0].src[s];
      for (int cb0 = 0; cb0 < w0.ninp / 16; cb0 += 2)
        for (size_t first = 0, round = 0; first == 0 || first < reds.size(); first += 2, round++) {
          ReduceBwdJob j{};
          j.s = s; j.fn = f; j.nin = w0.ninp; j.stride_out = w0.nfun; j.cb0 = cb0; j.nb = std::min(2, w0.ninp / 16 - cb0);
          j.ncon = (int) std::min<size_t>(2, reds.size() - first);
          j.w = (long long) vB.size();
          j.wmu = (long long) j.ncon * 2 * 8 * 64;
          vB.resize(vB.size() + (size_t) nel * j.wmu, (T) 0);
          for (int q = 0; q < j.ncon; q++) {
            const ReduceSpec &sp = specs[reds[first + q]];
            j.sel[q] = sp.sel; j.stride[q] = sp.ostride; j.off[q] = sp.ooff; j.nout[q] = sp.nout; j.nks[q] = (sp.nout + 3) / 4;
            for (int mu = 0; mu < nel; mu++) {
              reduce_matrix(sp.src[s], sp.fo, f, mu, sp.nout, M);
              for (int cb = 0; cb < j.nb; cb++)
                for (int k4 = 0; k4 < j.nks[q]; k4++)
                  for (int lane = 0; lane < 64; lane++) {
                    const int k = 4 * k4 + (lane >> 4), n = (cb0 + cb) * 16 + (lane & 15);
                    if (k < sp.nout && n < sp.src[s].n_in)
                      vB[(size_t) (j.w + mu * j.wmu + ((q * 2 + cb) * 8 + k4) * 64 + lane)] = (T) M[(size_t) n * sp.nout + k];
                  }
            }
          }
          auto put = [&](std::vector<std::unique_ptr<List>> &l) {
            while (l.size() <= round) l.emplace_back(new List());
            l[round]->host.push_back(j);
          };
          put(all);
          if (j.ncon > 0) put(s >= 2 ? high : low);
        }
    };
    for (const auto &kv : fed) add_rows(kv.first.first, kv.first.second, kv.second);
    for (size_t f = 0; f < cover.size(); f++)
      if (cover[f] && !fed.count({0, (int) f})) add_rows(0, (int) f, {});
    upload_vec(WB, vB);
    for (auto *l : {&high, &low, &all})
      for (auto &x : *l) upload_vec(x->dev, x->host);
  }
};

// Device, stream, per-stage GPU timing and the MFMA accumulator-row probe of an engine.
// First base of an engine: from its construction until end_build() every DevBuf made on this thread (members of the
// engine and of the structures it holds) is listed in bufs_, and what they allocate in that time is model data.
struct BufRegistry {
  std::vector<DevBuf *> bufs_;
  BufRegistry() { building_registry() = &bufs_; }
  ~BufRegistry()
  {
    if (building_registry() == &bufs_) building_registry() = nullptr;    // a constructor that threw
  }
  void end_build()
  {
    if (building_registry() == &bufs_) building_registry() = nullptr;
  }
};

class EngineBase : public Engine, protected BufRegistry {
 public:
  // Frees every buffer that was allocated after the engine was built (per-atom and per-bond work buffers, the uploaded
  // structure); weights, tables and compiled kernels stay.  The engine then holds no structure: upload before the next
  // run.  The reference's engines: release_buffers() (kk/grace_1l_kk.h:72-113).
  void release_buffers() override
  {
    HIP_CHECK(hipSetDevice(device_));
    HIP_CHECK(hipStreamSynchronize(stream_));
    for (DevBuf *b : bufs_)
      if (!b->model_data) b->release();
    have_sid_ = false;
    chunk_laid_out_ = 0;
    n_peak_ = 0;
    n_ = 0;
    n_nodes_ = 0;
    nb_ = 0;
    nstruct_ = 1;
    ran_ = ran_forces_ = ran_eatom_ = ran_uq_ = ran_vatom_ = false;
    upload_serial_++;
  }
  void synchronize() override { check(hipSetDevice(device_), "hipSetDevice"); check(hipStreamSynchronize(stream_), "hipStreamSynchronize"); }
  void set_chunksize(int atoms) override
  {
    if (!chunks_ && atoms > 0)
      throw InvalidArgument(who_ + ": this engine evaluates a structure in one pass; chunksize must be 0 (one pass) or -1 (auto), got " +
                            std::to_string(atoms));
    chunk_request_ = atoms;
  }
  int chunksize_used() const override { return chunk_used_; }
  void set_spline(int n) override
  {
    if (n < 0 || (n > 0 && n < 16) || n > (1 << 20)) throw InvalidArgument(who_ + ": spline must be 0 (the radial MLP itself) or 16 .. 1048576 intervals");
    apply_spline(n);
    spline_n_ = n;
  }
  int spline() const override { return spline_n_; }
  void set_ordered_sums(bool on) override
  {
    if (on && !ordered_ok_) throw InvalidArgument(who_ + ": this engine has no ordered (atomic-free) sums");
    ordered_ = on;
  }
  bool ordered_sums() const override { return ordered_; }
  void set_exchange(const ExchangeCallbacks &cb) override { exchange_ = cb; }
  int comm_layers() const override { return 0; }
  int comm_width(int) const override { return 0; }
  void comm_rows(int, int, int, const int *, int, double *, bool) override { throw Error(who_ + ": this model kind has no message rows to exchange"); }
  int64_t atoms_that_fit() override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (chunks_ && chunk_request_ < 0) return INT64_MAX;    // the engine splits a pass that does not fit by itself
    if (n_peak_ <= 0 || chunk_used_ > 0) return layers() == 3 ? 16384 : layers() == 2 ? 131072 : 262144;
    double held = 0.0;
    for (const DevBuf *b : bufs_)
      if (!b->model_data) held += (double) b->bytes;
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    double avail = (double) free_b + (double) device_pool().held_on(device_);
    const long long cap = dev_bytes_limit().load();
    if (cap > 0) avail = std::min(avail, (double) (cap - dev_bytes_in_use().load()));
    // the buffers grew to the largest pass since they were last released: that pass fits, and sets the bytes per atom
    const double per_atom = std::max(held / n_peak_, 1.0);
    return std::max<int64_t>(n_peak_, (int64_t) (0.7 * (avail + held) / per_atom));
  }
  void set_profile(bool on) override { profile_ = on; }
  const std::vector<StageTime> &stage_times() override
  {
    synchronize();
    times_.clear();
    for (size_t q = 0; q < ev_used_; q++) {
      float ms = 0.f;
      check(hipEventElapsedTime(&ms, events_[q].first, events_[q].second), "hipEventElapsedTime");
      auto it = std::find_if(times_.begin(), times_.end(), [&](const StageTime &s) { return s.name == ev_names_[q]; });
      if (it == times_.end()) {
        times_.push_back({ev_names_[q], 0.0, 0});
        it = times_.end() - 1;
      }
      it->ms += ms;
      it->launches++;
      it->flops += ev_flops_[q];
    }
    return times_;
  }
  void debug_copy(int64_t bytes) override
  {
    check(hipSetDevice(device_), "hipSetDevice");
    const long long nd = std::max<int64_t>(bytes / 8, 1);
    DevBuf a, b;
    a.ensure(nd * 8);
    b.ensure(nd * 8);
    check(hipMemsetAsync(a.p, 0, nd * 8, stream_), "hipMemsetAsync");
    hipLaunchKernelGGL(k_copy_calibration, dim3(4096), dim3(256), 0, stream_, a.as<double>(), b.as<double>(), nd);
    check(hipGetLastError(), "copy kernel");
    check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  }
  // GB/s of the copy kernel (bytes read + bytes written) and of a read-only stream kernel over `bytes` bytes, best of 5
  void stream_rates(int64_t bytes, double *copy_gbs, double *read_gbs) override
  {
    check(hipSetDevice(device_), "hipSetDevice");
    const long long nd = std::max<int64_t>(bytes / 16, 1) * 2;
    DevBuf a, b, part;
    a.ensure(nd * 8);
    b.ensure(nd * 8);
    part.ensure(4096 * 8);
    check(hipMemsetAsync(a.p, 0, nd * 8, stream_), "hipMemsetAsync");
    check(hipMemsetAsync(part.p, 0, 4096 * 8, stream_), "hipMemsetAsync");
    hipEvent_t e0, e1;
    check(hipEventCreate(&e0), "hipEventCreate");
    check(hipEventCreate(&e1), "hipEventCreate");
    double best[2] = {1e30, 1e30};
    for (int rep = 0; rep < 6; rep++)
      for (int k = 0; k < 2; k++) {
        check(hipEventRecord(e0, stream_), "hipEventRecord");
        if (k == 0) hipLaunchKernelGGL(k_copy_calibration, dim3(4096), dim3(256), 0, stream_, a.as<double>(), b.as<double>(), nd);
        else hipLaunchKernelGGL(k_read_calibration, dim3(4096), dim3(256), 0, stream_, a.as<double>(), part.as<double>(), nd);
        check(hipEventRecord(e1, stream_), "hipEventRecord");
        check(hipEventSynchronize(e1), "hipEventSynchronize");
        float ms = 0.f;
        check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
        if (rep > 0) best[k] = std::min(best[k], (double) ms);
      }
    (void) hipEventDestroy(e0);
    (void) hipEventDestroy(e1);
    if (copy_gbs) *copy_gbs = 2.0 * nd * 8 / (best[0] * 1e-3) * 1e-9;
    if (read_gbs) *read_gbs = 1.0 * nd * 8 / (best[1] * 1e-3) * 1e-9;
  }

  // copies a CSR structure to the device after the argument checks of the reference's CSR entry
  // (python/src/core.cpp:292-396); atoms are grouped into tiles of 16 of one element for the tile GEMMs
  void upload(const CsrInput &in) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (in.n < 0) throw InvalidArgument("negative atom count");
    const bool table = in.x && in.image && in.shifts;
    if ((in.rij != nullptr) == (in.x || in.image || in.shifts) || (!in.rij && !table))
      throw InvalidArgument("give rij or positions, image and shifts");
    const int n = in.n, nn = std::max(in.n, in.n_nodes);
    if (nn > n && (in.sid || !in.rij)) throw InvalidArgument("a list with ghost atoms holds one structure and gives its bond vectors");
    std::vector<int> mu(nn);
    for (int a = 0; a < nn; a++) {
      if (in.types[a] < 1 || in.types[a] > ntypes_) throw InvalidArgument("types must be 1 .. len(species)");
      mu[a] = type2mu_[in.types[a]];
      if (mu[a] < 0)
        throw Error(who_ + ": atom " + std::to_string(a) + " of unmapped type " + std::to_string(in.types[a]) + " in the atom list");
    }
    if (in.offset[0] != 0) throw InvalidArgument("offset[0] must be 0 and offset[-1] == len(j)");
    for (int a = 0; a < n; a++)
      if (in.offset[a + 1] < in.offset[a]) throw InvalidArgument("offset must be non-decreasing");
    const int64_t nb = in.offset[n];
    for (int64_t q = 0; q < nb; q++) {
      if (in.j[q] < 0 || in.j[q] >= nn) throw InvalidArgument("j must index atoms 0 .. len(types)-1");
      if (in.image && (in.image[q] < 0 || in.image[q] >= in.nimages)) throw InvalidArgument("image must index rows of shifts");
    }
    if (in.nstruct < 1) throw InvalidArgument("the number of structures must be positive");
    if (in.sid)
      for (int a = 0; a < n; a++)
        if (in.sid[a] < 0 || in.sid[a] >= in.nstruct) throw InvalidArgument("structure index of an atom out of range");
    if (in.sid)
      for (int a = 0; a < n; a++)
        for (int64_t q = in.offset[a]; q < in.offset[a + 1]; q++)
          if (in.sid[in.j[q]] != in.sid[a]) throw InvalidArgument("a bond joins atoms of two structures");
    HIP_CHECK(hipStreamSynchronize(stream_));
    n_ = n;
    n_nodes_ = nn;
    nb_ = nb;
    nstruct_ = in.sid ? in.nstruct : 1;
    have_sid_ = in.sid != nullptr;
    sid_sorted_ = !in.sid || std::is_sorted(in.sid, in.sid + n);
    have_rij_ = in.rij != nullptr;
    auto put = [&](DevBuf &b, const void *src, size_t bytes) {
      b.ensure(std::max<size_t>(bytes, 8));
      if (bytes) HIP_CHECK(hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, stream_));
    };
    put(mu_, mu.data(), sizeof(int) * nn);
    if (have_sid_) put(sid_, in.sid, sizeof(int) * n);
    mu_host_.assign(mu.begin(), mu.begin() + n);    // the central atoms: they make the element tiles
    chunk_laid_out_ = 0;
    const std::vector<int> tiles = element_tiles(mu_host_, nelem_, tile_el_);
    ntiles_ = (int) tiles.size() / 16;
    put(tiles_, tiles.data(), sizeof(int) * tiles.size());
    static_assert(sizeof(long long) == sizeof(int64_t), "offset type");
    put(offset_, in.offset, sizeof(int64_t) * (n + 1));
    put(j_, in.j, sizeof(int) * nb);
    if (have_rij_) put(rij_, in.rij, sizeof(double) * 3 * nb);
    else {
      put(x_, in.x, sizeof(double) * 3 * n);
      put(image_, in.image, sizeof(int) * nb);
      put(shifts_, in.shifts, sizeof(double) * 3 * in.nimages);
    }
    HIP_CHECK(hipStreamSynchronize(stream_));    // the host copies (mu, tiles) go out of scope
    ran_ = false;
    upload_serial_++;
  }
  void upload_device(const DeviceCsr &in) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (in.n < 0) throw InvalidArgument("negative atom count");
    const int n = in.n, nn = std::max(in.n, in.n_nodes);
    const bool vectors = in.rij || in.fill;
    if (nn > n && (in.sid || !vectors)) throw InvalidArgument("a list with ghost atoms holds one structure and gives its bond vectors");
    std::vector<int> mu(nn);
    for (int a = 0; a < nn; a++) {
      if (in.types[a] < 1 || in.types[a] > ntypes_) throw InvalidArgument("types must be 1 .. len(species)");
      mu[a] = type2mu_[in.types[a]];
      if (mu[a] < 0)
        throw Error(who_ + ": atom " + std::to_string(a) + " of unmapped type " + std::to_string(in.types[a]) + " in the atom list");
    }
    if (in.nstruct < 1) throw InvalidArgument("the number of structures must be positive");
    if (in.sid)
      for (int a = 0; a < n; a++)
        if (in.sid[a] < 0 || in.sid[a] >= in.nstruct) throw InvalidArgument("structure index of an atom out of range");
    HIP_CHECK(hipStreamSynchronize(stream_));
    if (in.fill) {    // first, so that the list is written while the host lays out the tiles
      j_.ensure(std::max<size_t>(sizeof(int) * (size_t) in.nb, 8));
      rij_.ensure(std::max<size_t>(sizeof(double) * 3 * (size_t) in.nb, 8));
      in.fill(j_.as<int>(), rij_.as<double>(), stream_);
    }
    n_ = n;
    n_nodes_ = nn;
    nb_ = in.nb;
    nstruct_ = in.sid ? in.nstruct : 1;
    have_sid_ = in.sid != nullptr;
    sid_sorted_ = !in.sid || std::is_sorted(in.sid, in.sid + n);
    have_rij_ = vectors;
    mu_host_.assign(mu.begin(), mu.begin() + n);    // the central atoms: they make the element tiles
    chunk_laid_out_ = 0;
    const std::vector<int> tiles = element_tiles(mu_host_, nelem_, tile_el_);
    ntiles_ = (int) tiles.size() / 16;
    auto put = [&](DevBuf &b, const void *src, size_t bytes, hipMemcpyKind kind) {
      b.ensure(std::max<size_t>(bytes, 8));
      if (bytes) HIP_CHECK(hipMemcpyAsync(b.p, src, bytes, kind, stream_));
    };
    put(mu_, mu.data(), sizeof(int) * nn, hipMemcpyHostToDevice);
    put(tiles_, tiles.data(), sizeof(int) * tiles.size(), hipMemcpyHostToDevice);
    put(offset_, in.offset, sizeof(int64_t) * (n + 1), hipMemcpyDeviceToDevice);
    if (have_sid_) put(sid_, in.sid, sizeof(int) * n, hipMemcpyHostToDevice);
    if (!in.fill) {
      put(j_, in.j, sizeof(int) * in.nb, hipMemcpyDeviceToDevice);
      if (have_rij_) put(rij_, in.rij, sizeof(double) * 3 * in.nb, hipMemcpyDeviceToDevice);
      else {
        put(image_, in.image, sizeof(int) * in.nb, hipMemcpyDeviceToDevice);
        put(x_, in.x, sizeof(double) * 3 * n, hipMemcpyDeviceToDevice);
        put(shifts_, in.shifts, sizeof(double) * 3 * in.nimages, hipMemcpyHostToDevice);
      }
    }
    HIP_CHECK(hipStreamSynchronize(stream_));
    ran_ = false;
    upload_serial_++;
  }
  void update_positions(const double *x) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (have_rij_) throw Error("update_positions: the uploaded list holds bond vectors, not positions");
    HIP_CHECK(hipStreamSynchronize(stream_));    // no pass of the stream still reads the staging memory or x_
    if (n_ > 0) {
      const size_t bytes = sizeof(double) * 3 * (size_t) n_;
      pin_in_.ensure(bytes);
      std::memcpy(pin_in_.p, x, bytes);
      HIP_CHECK(hipMemcpyAsync(x_.p, pin_in_.p, bytes, hipMemcpyHostToDevice, stream_));    // ordered before the pass on the same stream
    }
    ran_ = false;
  }
  double *bond_vectors_device() override
  {
    if (!have_rij_) throw Error("bond_vectors_device: the uploaded list holds positions, not bond vectors");
    HIP_CHECK(hipSetDevice(device_));
    HIP_CHECK(hipStreamSynchronize(stream_));
    ran_ = false;
    return rij_.as<double>();
  }
  uint64_t upload_serial() const override { return upload_serial_; }
  int device_index() const override { return device_; }
  void radial_noalloc(int, const double *, const int *, double *, double *) override
  {
    throw Error(who_ + ": the radial call without allocations is available for GRACE-1L engines");
  }
  // tiles of 16 atoms of one element (-1 padded), in atom order within an element, elements ascending;
  // el_off[e] .. el_off[e + 1]: the tiles of element e
  static std::vector<int> element_tiles(const std::vector<int> &mu, int nel, std::vector<int> &el_off)
  {
    // a counting pass per element (the elements are few): atoms per element, the tiles each element needs, then every atom
    // to the next free slot of its element, in atom order
    const int n = (int) mu.size();
    std::vector<int> count((size_t) nel, 0);
    for (int a = 0; a < n; a++) {
      if (mu[a] < 0 || mu[a] >= nel) throw Error("element of a central atom out of range");
      count[(size_t) mu[a]]++;
    }
    el_off.assign(nel + 1, 0);
    for (int e = 0; e < nel; e++) el_off[e + 1] = el_off[e] + (count[(size_t) e] + 15) / 16;
    std::vector<int> tiles((size_t) 16 * el_off[nel], -1), next((size_t) nel);
    for (int e = 0; e < nel; e++) next[(size_t) e] = 16 * el_off[e];
    for (int a = 0; a < n; a++) tiles[(size_t) next[(size_t) mu[a]]++] = a;
    return tiles;
  }
  void fetch(double *energy, double *forces, double *virial, double *eatom) override
  {
    if (have_sid_) throw Error("the uploaded list holds several structures: use fetch_batch()");
    fetch_batch(1, energy, forces, virial, eatom);
  }
  void fetch_batch(int nstruct, double *energy, double *forces, double *virial, double *eatom) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (!ran_) throw Error("fetch() before run()");
    if (nstruct != nstruct_) throw InvalidArgument("fetch_batch: the uploaded list holds " + std::to_string(nstruct_) + " structures");
    // everything the call returns goes to pinned memory as asynchronous copies behind the pass, with one wait:
    // [records 8 records()][forces 3 n_nodes][per-atom energies n]; the pass leaves its zero-bond flag in pin_flag_
    const bool wf = forces && ran_forces_ && n_nodes_ > 0, we = eatom && ran_eatom_ && n_ > 0;
    const size_t nrec = (size_t) 8 * records(), nf = wf ? (size_t) 3 * n_nodes_ : 0, ne = we ? (size_t) n_ : 0;
    pin_out_.ensure((nrec + nf + ne) * sizeof(double));
    double *rec = pin_out_.as<double>(), *pf = rec + nrec, *pe = pf + nf;
    HIP_CHECK(hipMemcpyAsync(rec, out_.p, (nrec + nf) * sizeof(double), hipMemcpyDeviceToHost, stream_));    // the forces stand behind the records
    if (we) HIP_CHECK(hipMemcpyAsync(pe, eatom_.p, ne * sizeof(double), hipMemcpyDeviceToHost, stream_));
    HIP_CHECK(hipStreamSynchronize(stream_));
    check_zero_bond();
    for (int q = 0; q < nstruct_; q++) {
      double s[7];
      add_records(rec, q, s);
      if (energy) energy[q] = s[0];
      if (virial && ran_forces_)
        for (int k = 0; k < 6; k++) virial[6 * (size_t) q + k] = s[1 + k];
    }
    if (wf) std::memcpy(forces, pf, nf * sizeof(double));
    if (we) std::memcpy(eatom, pe, ne * sizeof(double));
  }
  void fetch_batch_device(int nstruct, double *energy, double *forces, double *virial, double *eatom) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (!ran_) throw Error("fetch() before run()");
    if (nstruct != nstruct_) throw InvalidArgument("fetch_batch: the uploaded list holds " + std::to_string(nstruct_) + " structures");
    HIP_CHECK(hipStreamSynchronize(stream_));
    check_zero_bond();    // before anything is written to the caller's arrays
    hipLaunchKernelGGL(k_unpack_records, dim3((unsigned) ((nstruct_ + 255) / 256)), dim3(256), 0, stream_, scal_.as<double>(), nstruct_, record_copies(), energy,
                       ran_forces_ ? virial : nullptr);
    if (forces && ran_forces_ && n_ > 0) HIP_CHECK(hipMemcpyAsync(forces, f_.p, sizeof(double) * 3 * n_, hipMemcpyDeviceToDevice, stream_));
    if (eatom && ran_eatom_ && n_ > 0) HIP_CHECK(hipMemcpyAsync(eatom, eatom_.p, sizeof(double) * n_, hipMemcpyDeviceToDevice, stream_));
    HIP_CHECK(hipStreamSynchronize(stream_));
  }
  // two atoms at one position make a bond of length 0 (bonds.h:49-62 of the reference): reported by the pass in pin_flag_
  void check_zero_bond()
  {
    if (n_ == 0) return;
    // k_edge_fill writes it to the pinned memory itself; every caller has waited for the stream
    const int *zb = pin_flag_.as<int>();
    if (!zb) return;
    if (zb[0] >= 0)
      throw Error("two atoms at the same position (a bond of length 0 between atoms " + std::to_string(zb[0]) + " and " + std::to_string(zb[1]) +
                  " of the neighbour list): not a physical structure");
  }
  void fetch_add_device(const int *atom, double *energy, double *forces, double *virial, double *eatom) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (!ran_) throw Error("fetch() before run()");
    if (have_sid_) throw Error("the uploaded list holds several structures: use fetch_batch()");
    HIP_CHECK(hipStreamSynchronize(stream_));
    check_zero_bond();    // before anything is added to the caller's arrays
    const bool wf = forces && ran_forces_, we = eatom && ran_eatom_;
    if (n_nodes_ > n_ && atom) throw Error("fetch_add_device: a list with ghost atoms keeps the caller's atom order");
    if (n_ > 0 && (wf || we))
      hipLaunchKernelGGL(k_add_results, dim3((unsigned) ((n_nodes_ + 255) / 256)), dim3(256), 0, stream_, atom, n_nodes_, n_, f_.as<double>(),
                         wf ? forces : nullptr, eatom_.as<double>(), we ? eatom : nullptr);
    pin_out_.ensure((size_t) 8 * records() * sizeof(double));
    HIP_CHECK(hipMemcpyAsync(pin_out_.p, scal_.p, (size_t) 8 * records() * sizeof(double), hipMemcpyDeviceToHost, stream_));
    HIP_CHECK(hipStreamSynchronize(stream_));
    double s[7];
    add_records(pin_out_.as<double>(), 0, s);
    if (energy) *energy = s[0];
    if (virial && ran_forces_)
      for (int k = 0; k < 6; k++) virial[k] = s[1 + k];
  }
  void fetch_vatom(double *vatom, int ncomp, long long expect_rows = -1) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (ncomp != 6 && ncomp != 9) throw InvalidArgument("per-atom virials have 6 or 9 components");
    if (!ran_ || !ran_vatom_) throw Error("fetch_vatom() needs a run with the per-atom virial flag (and forces)");
    if (expect_rows >= 0 && expect_rows != n_nodes_)
      throw Error("fetch_vatom(): the engine holds " + std::to_string(n_nodes_) + " rows, the caller expects " + std::to_string(expect_rows));
    HIP_CHECK(hipStreamSynchronize(stream_));
    check_zero_bond();
    if (!vatom || n_nodes_ <= 0) return;
    std::vector<double> rows((size_t) 9 * n_nodes_);
    HIP_CHECK(hipMemcpy(rows.data(), vatom_.p, sizeof(double) * rows.size(), hipMemcpyDeviceToHost));
    for (size_t q = 0; q < (size_t) n_nodes_; q++)
      for (int k = 0; k < ncomp; k++) vatom[(size_t) ncomp * q + k] = rows[9 * q + k];
  }
  void add_vatom_device(const int *atom, double *vatom, int ncomp) override
  {
    if (ncomp != 6 && ncomp != 9) throw InvalidArgument("per-atom virials have 6 or 9 components");
    HIP_CHECK(hipSetDevice(device_));
    if (!ran_ || !ran_vatom_) throw Error("per-atom virials need a run with the per-atom virial flag (and forces)");
    if (n_nodes_ > n_ && atom) throw Error("add_vatom_device: a list with ghost atoms keeps the caller's atom order");
    HIP_CHECK(hipStreamSynchronize(stream_));
    check_zero_bond();
    const long long tot = (long long) ncomp * n_nodes_;
    if (tot > 0)
      hipLaunchKernelGGL(k_add_rows, dim3((unsigned) ((tot + 255) / 256)), dim3(256), 0, stream_, atom, n_nodes_, (const double *) vatom_.as<double>(), 9,
                         ncomp, vatom);
    HIP_CHECK(hipStreamSynchronize(stream_));
  }
  void fetch_uq(double *gamma, double *sigma, double *cluster) override
  {
    HIP_CHECK(hipSetDevice(device_));
    if (!ran_ || !ran_uq_) throw Error("fetch_uq() needs a run with the UQ flag");
    HIP_CHECK(hipStreamSynchronize(stream_));
    if (n_ == 0) return;
    // host or device destinations (the batch call on device arrays hands in device pointers)
    if (gamma) HIP_CHECK(hipMemcpy(gamma, uq_gamma_.p, sizeof(double) * n_, hipMemcpyDefault));
    if (sigma) HIP_CHECK(hipMemcpy(sigma, uq_sigma_.p, sizeof(double) * n_, hipMemcpyDefault));
    if (cluster) HIP_CHECK(hipMemcpy(cluster, uq_cluster_.p, sizeof(double) * n_, hipMemcpyDefault));
  }
  int64_t last_edge_count() override
  {
    synchronize();
    long long e = 0;
    if (n_ > 0) HIP_CHECK(hipMemcpy(&e, eoff_.as<long long>() + n_, sizeof(e), hipMemcpyDeviceToHost));
    return e;
  }
  int64_t last_radial_rows() override
  {
    if (n_ == 0 || !paired_) return last_edge_count();
    synchronize();
    std::vector<long long> rows((size_t) pair_chunks_);
    HIP_CHECK(hipMemcpy(rows.data(), nrows_.p, rows.size() * sizeof(long long), hipMemcpyDeviceToHost));
    return std::accumulate(rows.begin(), rows.end(), 0ll);
  }
  double cutoff(int t1, int t2) const override
  {
    if (t1 < 1 || t1 > ntypes_ || t2 < 1 || t2 > ntypes_) return 0.0;
    const int a = type2mu_[t1], b = type2mu_[t2];
    return (a < 0 || b < 0) ? 0.0 : cut_host_[(size_t) a * nelem_ + b];
  }
  double max_cutoff() const override
  {
    double m = 0.0;
    for (int a = 1; a <= ntypes_; a++)
      for (int b = 1; b <= ntypes_; b++) m = std::max(m, cutoff(a, b));
    return m;
  }

 protected:
  // pair cutoffs [nel][nel] of the model
  void set_cutoffs(const std::vector<double> &cut)
  {
    cut_host_ = cut;
    upload_vec(cut_, cut);
  }
  // start of a pass: clears the outputs, filters the bonds of the uploaded list (r^2 < rc^2, bonds.h:120-162 of the
  // reference) into the compact edge arrays.  false: no atoms, nothing to do.
  bool begin_pass(const RunFlags &fl)
  {
    HIP_CHECK(hipSetDevice(device_));
    // argument checks first: a refused call leaves the state of the last good run (fetch() after it returns that run)
    if (fl.uq && !has_uq_head_) throw InvalidArgument(who_ + ": the model has no usable UQ head (" + uq_why_ + ")");
    ev_used_ = 0;
    const int n = n_;
    PassClear clear{};
    clear.nout = (long long) (8 * records()) + 3ll * n_nodes_;
    out_.ensure((size_t) clear.nout * sizeof(double));
    clear.out = scal_.p = out_.as<double>();
    f_.p = scal_.p + 8 * records();
    eatom_.ensure(std::max<size_t>(n, 1) * sizeof(double));
    ran_ = true;
    n_peak_ = std::max(n_peak_, n_);
    ran_forces_ = !fl.energy_only;
    ran_vatom_ = fl.vatom && !fl.energy_only;
    if (ran_vatom_) {
      clear.nvatom = 9ll * n_nodes_;
      vatom_.ensure((size_t) std::max<long long>(clear.nvatom, 1) * sizeof(double));
      clear.vatom = vatom_.as<double>();
    }
    ran_eatom_ = fl.eatom;
    ran_uq_ = false;    // set by the engine that evaluates a UQ head
    if (n == 0) {
      HIP_CHECK(hipMemsetAsync(clear.out, 0, (size_t) clear.nout * sizeof(double), stream_));
      if (clear.nvatom) HIP_CHECK(hipMemsetAsync(clear.vatom, 0, (size_t) clear.nvatom * sizeof(double), stream_));
      return false;
    }
    clear.zero_bond = zero_.as<int>();
    // no pass with other bonds is in flight: whatever changes the list or the positions has waited for the stream
    pin_flag_.ensure(2 * sizeof(int));
    pin_flag_.as<int>()[0] = pin_flag_.as<int>()[1] = -1;
    count_.ensure(sizeof(int) * n);
    eoff_.ensure(sizeof(long long) * (n + 1));
    BondSrc src{};
    src.mu = mu_.as<int>(); src.offset = offset_.as<long long>(); src.j = j_.as<int>();
    src.rij = have_rij_ ? rij_.as<double>() : nullptr;
    src.x = have_rij_ ? nullptr : x_.as<double>();
    src.image = have_rij_ ? nullptr : image_.as<int>();
    src.shifts = have_rij_ ? nullptr : shifts_.as<double>();
    src.cut = cut_.as<double>(); src.nel = nelem_;
    const size_t ecap = (size_t) std::max<int64_t>(nb_, 1);
    ei_.ensure(ecap * sizeof(int)); ej_.ensure(ecap * sizeof(int)); emu_.ensure(ecap * sizeof(int));
    rh_.ensure(ecap * 3 * sizeof(double)); r_.ensure(ecap * sizeof(double)); xr_.ensure(ecap * sizeof(double));
    rc_.ensure(ecap * sizeof(double));
    Edges ed{ei_.as<int>(), ej_.as<int>(), emu_.as<int>(), rh_.as<double>(), r_.as<double>(), xr_.as<double>(), rc_.as<double>(), nullptr};
    want_pairs_ = want_pairs_ && nb_ > 0 && nb_ < INT32_MAX;
    if (want_pairs_) {
      erow_.ensure(ecap * sizeof(int));
      ed.erow = erow_.as<int>();
    }
    const dim3 grid((unsigned) ((n + 3) / 4)), block(256);
    stage("edge_count", [&] { hipLaunchKernelGGL(k_edge_count, grid, block, 0, stream_, src, n, count_.as<int>(), clear); });
    const bool scan = n > kFillScanAtoms;
    if (scan) stage("edge_scan", [&] { launch_scan(stream_, count_.as<int>(), n, eoff_.as<long long>()); });
    stage("edge_fill", [&] {
      hipLaunchKernelGGL(scan ? k_edge_fill<false> : k_edge_fill<true>, grid, block, 0, stream_, src, n, (const int *) count_.as<int>(),
                         eoff_.as<long long>(), ed, zero_.as<int>(), pin_flag_.as<int>());
    });
    return true;
  }
  EngineBase(int device, const char *who, int ntypes, const std::vector<int> &type2mu, int n_elements) :
      device_(device), who_(who), ntypes_(ntypes), type2mu_(type2mu), nelem_(n_elements)
  {
    check_type2mu(type2mu_, ntypes_, n_elements, who);
    check(hipSetDevice(device_), "hipSetDevice");
    hipDeviceProp_t prop;
    check(hipGetDeviceProperties(&prop, device_), "hipGetDeviceProperties");
    if (std::string(prop.gcnArchName).rfind("gfx950", 0) != 0 && std::string(prop.gcnArchName).rfind("gfx942", 0) != 0)
      throw Error(std::string(who) + ": this library is built for gfx950 (MI355X); device is " + prop.gcnArchName);
    ncu_ = prop.multiProcessorCount;
    arch_ = prop.gcnArchName;
    check(hipStreamCreate(&stream_), "hipStreamCreate");
    zero_.ensure(2 * sizeof(int));
  }
  ~EngineBase() override
  {
    (void) hipSetDevice(device_);
    for (auto &e : events_) { (void) hipEventDestroy(e.first); (void) hipEventDestroy(e.second); }
    if (stream_) (void) hipStreamDestroy(stream_);
  }
  static void check(hipError_t e, const char *what)
  {
    if (e != hipSuccess) throw Error(std::string("HIP error: ") + hipGetErrorString(e) + " in " + what);
  }
  void prof_begin(const char *name)
  {
    if (!profile_) return;
    if (ev_used_ == events_.size()) {
      hipEvent_t a, b;
      check(hipEventCreate(&a), "hipEventCreate");
      check(hipEventCreate(&b), "hipEventCreate");
      events_.push_back({a, b});
      ev_names_.push_back("");
      ev_flops_.push_back(0.0);
    }
    cur_flops_ = 0.0;
    ev_names_[ev_used_] = name;
    check(hipEventRecord(events_[ev_used_].first, stream_), "hipEventRecord");
  }
  void prof_end()
  {
    if (!profile_) return;
    check(hipEventRecord(events_[ev_used_].second, stream_), "hipEventRecord");
    ev_flops_[ev_used_] = cur_flops_;
    ev_used_++;
  }
  template<class F> void stage(const char *name, F &&f)
  {
    prof_begin(name);
    f();
    check(hipGetLastError(), name);
    prof_end();
  }
  // which accumulator row each (lane / 16, register) of a 16x16x4 MFMA holds; the column must be lane % 16
  template<class T> void probe_mfma()
  {
    std::vector<T> A(64), B(64), D(256);
    for (int i = 0; i < 16; i++)
      for (int k = 0; k < 4; k++) {
        A[i * 4 + k] = (T) (1 + i + 16 * k);
        B[k * 16 + i] = (T) ((k == 0 ? 1 : k == 1 ? 3 : k == 2 ? 7 : 11) * (i + 1));
      }
    DevBuf dA, dB, dD;
    upload_vec(dA, A);
    upload_vec(dB, B);
    dD.ensure(256 * sizeof(T));
    hipLaunchKernelGGL(k_mfma_probe<T>, dim3(1), dim3(64), 0, stream_, dA.as<T>(), dB.as<T>(), dD.as<T>());
    check(hipGetLastError(), "k_mfma_probe");
    check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
    check(hipMemcpy(D.data(), dD.p, 256 * sizeof(T), hipMemcpyDeviceToHost), "hipMemcpy");
    double ref[16][16];
    for (int i = 0; i < 16; i++)
      for (int j = 0; j < 16; j++) {
        double s = 0;
        for (int k = 0; k < 4; k++) s += (double) A[i * 4 + k] * (double) B[k * 16 + j];
        ref[i][j] = s;
      }
    for (int g = 0; g < 4; g++)
      for (int v = 0; v < 4; v++) {
        int row = -1;
        for (int i = 0; i < 16 && row < 0; i++) {
          bool ok = true;
          for (int c = 0; c < 16 && ok; c++) ok = (double) D[(g * 16 + c) * 4 + v] == ref[i][c];
          if (ok) row = i;
        }
        if (row < 0) throw Error("MFMA 16x16x4 accumulator layout of this device is not the one the kernels assume");
        drow_[g * 4 + v] = row;
      }
    int seen = 0;    // the 16 (group, register) pairs must cover the 16 rows
    for (int q = 0; q < 16; q++) seen |= 1 << drow_[q];
    if (seen != 0xFFFF) throw Error("MFMA 16x16x4 accumulator layout probe failed");
  }
  // A[atom][lm][n] = sum over the atom's edges of Y_lm Rz_l[n]: on the matrix cores where the register tiles fit
  // (PAIRS: the engine may pair the radial rows)
  template<class T, bool PAIRS> void launch_scatter(ScatterArgs<T> sa, int n, int lmax)
  {
    sa.natoms = n;
    for (int q = 0; q < 16; q++) sa.drow[q] = drow_[q];
    const int kb = sa.C / 16;
    const size_t lds = (size_t) 4 * scatter_harmonics(sa.nl) * sa.nlm * sizeof(T);
    const dim3 grid((n + 3) / 4), block(256);
#define GR_SCAT(NL_, KB_)                                                                       \
  do {                                                                                          \
    auto kern = sa.tb.F ? k_scatter_a_tab<T, NL_, KB_> : k_scatter_a_mfma<T, NL_, KB_, RowsOf::bonds>; \
    if constexpr (PAIRS) if (sa.erow) kern = k_scatter_a_mfma<T, NL_, KB_, RowsOf::pairs>;      \
    hipLaunchKernelGGL(kern, grid, block, lds, stream_, sa);                                    \
  } while (0)
    const int key = sa.nl * 10 + kb;    // register tiles of the kernel: nl * kb <= 10
    if (key == 11) GR_SCAT(1, 1); else if (key == 12) GR_SCAT(1, 2); else if (key == 14) GR_SCAT(1, 4);
    else if (key == 21) GR_SCAT(2, 1); else if (key == 22) GR_SCAT(2, 2); else if (key == 24) GR_SCAT(2, 4);
    else if (key == 31) GR_SCAT(3, 1); else if (key == 32) GR_SCAT(3, 2);
    else if (key == 41) GR_SCAT(4, 1); else if (key == 42) GR_SCAT(4, 2);
    else if (key == 51) GR_SCAT(5, 1); else if (key == 52) GR_SCAT(5, 2);
    else if (key == 61) GR_SCAT(6, 1); else if (key == 71) GR_SCAT(7, 1);
#undef GR_SCAT
    else {
      if (sa.tb.F) throw Error("A basis from radial tables: the channel widths of this model have no matrix-core kernel");
      const int sthreads = round_up(sa.nl * sa.C, 64);
      auto kern = lmax <= 4 ? k_scatter_a<T, 9, RowsOf::bonds> : k_scatter_a<T, 13, RowsOf::bonds>;
      if constexpr (PAIRS) if (sa.erow) kern = lmax <= 4 ? k_scatter_a<T, 9, RowsOf::pairs> : k_scatter_a<T, 13, RowsOf::pairs>;
      hipLaunchKernelGGL(kern, dim3(n), dim3(sthreads), 0, stream_, sa);
    }
  }
  // per-bond forces of a layer from the adjoint of its A basis (k_bond_bwd); ba.drow is filled here
  template<class T, bool PAIRS> void launch_bond_bwd(BondBwdArgs<T> ba, int n)
  {
    for (int q = 0; q < 16; q++) ba.drow[q] = drow_[q];
    ba.tiles = bond_bwd_tiles<T>(!one_order() && n <= 2 * ncu_);
    const int kb = ba.C / 16;
    const size_t lds = ((size_t) ba.nlm * (ba.C + 2) + (size_t) 4 * 16 * bond_bwd_row(ba.nlm)) * sizeof(T);      // four tiles of bonds
    if (kb != 1 && kb != 2 && kb != 4) throw Error("bond backward: channel width must be 16, 32 or 64");
    if (ba.tb.F && ba.noutp != ba.nl * ba.C) throw Error("bond backward: rows of the radial tables of another width");
#define GR_BB(KB, NL)                                                                                  \
  do {                                                                                                 \
    auto kern = ba.tb.F ? k_bond_bwd<T, KB, NL, RowsOf::tables> : k_bond_bwd<T, KB, NL, RowsOf::bonds>; \
    if constexpr (PAIRS) if (ba.erow) kern = k_bond_bwd<T, KB, NL, RowsOf::pairs>;                     \
    hipLaunchKernelGGL(kern, dim3(n), dim3(256 / ba.tiles), lds, stream_, ba);                          \
  } while (0)
#define GR_BB_NL(NL) case NL: if (kb == 1) GR_BB(1, NL); else if (kb == 2) GR_BB(2, NL); else GR_BB(4, NL); break
    switch (ba.nl) {
      GR_BB_NL(1); GR_BB_NL(2); GR_BB_NL(3); GR_BB_NL(4); GR_BB_NL(5); GR_BB_NL(6); GR_BB_NL(7);
      default: throw Error("bond backward: lmax above " + std::to_string(kKernMaxL));
    }
#undef GR_BB_NL
#undef GR_BB
  }
  // With ordered sums a GRACE-1L result does not depend on the chunk size: kernels whose sums have another order are then not
  // chosen by the number of atoms of a pass (k_gemm_few deals the segments of a job to four waves, chain_bwd_part the groups of
  // a chain to several blocks, k_bond_bwd in fp32 the tiles of an atom's bonds to two waves or four).
  bool one_order() const { return ordered_ && layers() == 1; }
  // Which launches with one input width take k_gemm_few / k_gemm_wide: all of 64 x 64 channels, and those whose blocks of
  // k_gemm_jobs (16 atom tiles each) would leave CUs idle.
  bool gemm_io_shape(int njobs, int kb, int nb, int ntiles) const
  {
    return (kb == 4 && nb == 4) || (!one_order() && (long long) njobs * ((ntiles + 15) / 16) < ncu_);
  }
  // Which launches of 64 x 64 channels take k_gemm_wide: where groups of eight atom tiles (a block in fp64, two in fp32) fill
  // the chip twice, or half of it when the jobs are long enough for its better use of the weights to count.  Measured,
  // k_gemm_few / k_gemm_wide, 36 jobs: one segment, 190 tiles (864 groups, fp64) 51 / 36 us; 47 segments, 8 tiles (36 groups)
  // 25 / 50, 47 tiles 42 / 35, 190 tiles 369 / 185.  fp32 with the line at half as many tiles: the pass of 150 atoms
  // 3.34 -> 3.43 ms, of 200 atoms 3.70 -> 3.77, from 300 atoms on the same.
  template<class T> bool gemm_wide_shape(const DevJobs<T> &J, int ntiles) const
  {
    return one_order() || (long long) J.d.njobs * ((ntiles + 7) / 8) >= (J.seg_count >= 4ll * J.d.njobs ? ncu_ / 2 : 2 * ncu_);
  }
  template<class T> void launch_gemm_io(DevJobs<T> &J, int kb, int nb, const GemmIO<T> &io, const int *tiles, int ntiles)
  {
    if (J.d.njobs == 0 || ntiles == 0) return;
    cur_flops_ += 2.0 * 16.0 * ntiles * (double) (nb * 16) * (double) (kb * 16) * (double) J.seg_count;
    if (kb == 4 && nb == 4 && !J.d.job_add && gemm_wide_shape(J, ntiles)) {
      constexpr int group = 4 * gemm_wide_tiles<T>();    // atom tiles of a block
      const int groups = (ntiles + group - 1) / group;
      const int reps = J.d.max_seg == 1 && !io.accumulate ? std::max(1, std::min(8, (int) ((long long) J.d.njobs * groups / (8 * ncu_)))) : 1;
      hipLaunchKernelGGL(k_gemm_wide<T>, dim3(J.d.njobs, (groups + reps - 1) / reps), dim3(256), 0, stream_, J.d, io, tiles, ntiles, reps);
      return;
    }
    const dim3 grid(J.d.njobs, ntiles);
#define GR_FEW(K_, N_)                                                                                                              \
  {                                                                                                                                 \
    if (J.d.max_seg >= 4) hipLaunchKernelGGL((k_gemm_few<T, K_, N_, 4>), grid, dim3(64 * N_ * 4), 0, stream_, J.d, io, tiles);      \
    else hipLaunchKernelGGL((k_gemm_few<T, K_, N_, 1>), grid, dim3(64 * N_), 0, stream_, J.d, io, tiles);                           \
  }
    switch (kb * 10 + nb) {
      case 11: GR_FEW(1, 1) break;
      case 12: GR_FEW(1, 2) break;
      case 14: GR_FEW(1, 4) break;
      case 21: GR_FEW(2, 1) break;
      case 22: GR_FEW(2, 2) break;
      case 24: GR_FEW(2, 4) break;
      case 41: GR_FEW(4, 1) break;
      case 42: GR_FEW(4, 2) break;
      case 44: GR_FEW(4, 4) break;
      default: throw Error("unsupported channel widths");
    }
#undef GR_FEW
  }
  // out[tile atoms][job output] = GEMM jobs over X0 (kb0 16-channel blocks) and X1 (kb1), nb output blocks
  static constexpr size_t kGemmLdsBudget = 24 * 1024;    // measured on the benchmarks: 24 kB beats 16, 40 and 64 kB (blocks per CU)
  template<class T>
  void launch_gemm(DevJobs<T> &J, int kb0, int kb1, int nb, const T *X0, int nf0, const T *X1, int nf1, T *out, int nfo, int accumulate,
                   const int *tiles, int ntiles)
  {
    if (J.d.njobs == 0 || ntiles == 0) return;
    if (kb0 == kb1 && gemm_io_shape(J.d.njobs, kb0, nb, ntiles)) {
      GemmIO<T> io{};
      io.X[0] = X0; io.X[1] = X1; io.nf[0] = nf0; io.nf[1] = nf1; io.WF[0] = J.d.WF0; io.WF[1] = J.d.WF1;
      io.out[0] = out; io.nfo[0] = nfo; io.accumulate = accumulate ? 1 : 0;
      return launch_gemm_io<T>(J, kb0, nb, io, tiles, ntiles);
    }
    // multiply-adds of the launch: every segment is a [16 atoms x K] . [K x N] product per atom tile
    cur_flops_ += 2.0 * 16.0 * ntiles * (double) (nb * 16) * ((double) J.nseg[0] * kb0 * 16 + (double) J.nseg[1] * kb1 * 16);
    const int ksm = std::max(kb0, kb1) * 4;
    // weight tiles staged at a time: as many as fit kGemmLdsBudget, so that the wide tiles of 64-channel models (32 kB
    // in fp64) leave room for several blocks per CU
    const size_t tile_bytes = (size_t) nb * ksm * 64 * sizeof(T);
    const int mseg = std::max(1, std::min(kGemmMaxSeg, (int) (kGemmLdsBudget / tile_bytes)));
    const size_t lds = (size_t) mseg * tile_bytes;
    // single-segment jobs (one weight tile each: projections, reverse of the product reduces) walk several groups of
    // atom tiles per block when the grid is large: the staging of the tile is what they spend their time on
    // waves of a block: a staged weight set is shared by 8 waves at fp64, by 4 at fp32 (measured: 8 instead of 4 gives
    // -1.3 % of a pass on the fp64 benchmarks, +1.8 % at fp32)
    const int nwave = sizeof(T) == 8 ? 8 : 4;
    const int groups = (ntiles + nwave * kGemmTilesPerWave - 1) / (nwave * kGemmTilesPerWave);
    const int reps = J.d.max_seg == 1 ? std::max(1, std::min(8, (int) ((long long) J.d.njobs * groups / 8192))) : 1;
    const dim3 grid(J.d.njobs, (groups + reps - 1) / reps);
#define GR_GEMM(A_, B_, C_)                                                                                            \
  {                                                                                                                    \
    auto kern = k_gemm_jobs<T, A_, B_, C_>;                                                                            \
    if (lds > 48 * 1024)                                                                                               \
      HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds)); \
    hipLaunchKernelGGL(kern, grid, dim3(64 * nwave), lds, stream_, J.d, X0, nf0, X1, nf1, out, nfo, tiles, ntiles, accumulate, reps, mseg); \
  }
#define GR_GEMM_C(A_, B_)                                                                                              \
  switch (nb) {                                                                                                        \
    case 1: GR_GEMM(A_, B_, 1) break;                                                                                  \
    case 2: GR_GEMM(A_, B_, 2) break;                                                                                  \
    case 4: GR_GEMM(A_, B_, 4) break;                                                                                  \
    default: throw Error("unsupported channel widths");                                                                \
  }
    switch (kb0 * 10 + kb1) {
      case 11: GR_GEMM_C(1, 1) break;
      case 12: GR_GEMM_C(1, 2) break;
      case 14: GR_GEMM_C(1, 4) break;
      case 21: GR_GEMM_C(2, 1) break;
      case 22: GR_GEMM_C(2, 2) break;
      case 24: GR_GEMM_C(2, 4) break;
      case 41: GR_GEMM_C(4, 1) break;
      case 42: GR_GEMM_C(4, 2) break;
      case 44:    // 64 outputs: k_gemm_few, k_gemm_wide
        if (nb == 1) { GR_GEMM(4, 4, 1) } else if (nb == 2) { GR_GEMM(4, 4, 2) } else throw Error("unsupported channel widths");
        break;
      default: throw Error("unsupported channel widths");
    }
#undef GR_GEMM_C
#undef GR_GEMM
  }

  // ---- the generated chain kernels (ChainKernels, jit_chain.hpp) over n atoms, in parts where n is small (parts_for) ----
  // Measured, GRACE-1L with 128 atoms (5 parts): forward 69 -> 32 us, reverse 87 -> 43 us with the sum of the parts;
  // GRACE-2L with 107 atoms: the four launches 51 + 52 + 58 + 62 -> 19 + 21 + 30 + 29 us (37 + 47 since P3 of layer 1, two launches of
  // 34 + 38 us, is inside them).
  template<class T, class K>
  void launch_chain_fwd(K &ck, int n, const T *X0, T *X1, T *P2, T *P21, T *P22, T *P3, T *P4, const T *W)
  {
    int nat = n, one = 1;
    const int np = one_order() ? 1 : ck.parts_for(n, ncu_);
    std::vector<void *> args = {&X0, &X1, &P2, &P21, &P22, &P3, &P4, &W, &nat, &one};
    if (np > 1)
      for (unsigned long long &m : ck.parts[np].mask) args.push_back(&m);
    const unsigned blocks = (unsigned) ((n + ck.atoms_per_block - 1) / ck.atoms_per_block);
    HIP_CHECK(hipModuleLaunchKernel(np > 1 ? ck.fwd_part : ck.fwd, blocks, np, 1, 256, 1, 1, 0, stream_, args.data(), nullptr));
    cur_flops_ += ck.flops_per_atom * n;
  }
  // returns the parts; with more than one launch_chain_sum() has to follow
  template<class T, class K>
  int launch_chain_bwd(K &ck, int n, const T *X0, const T *X1, const T *P21, const T *P22, const T *g2, const T *g3, const T *g4, const T *g21, T *gX0,
                        const T *W)
  {
    int nat = n, one = 1;
    const int np = one_order() ? 1 : ck.parts_for(n, ncu_);
    const unsigned blocks = (unsigned) ((n + ck.atoms_per_block - 1) / ck.atoms_per_block);
    long long stride = (long long) blocks * ck.atoms_per_block * ck.nf0 * ck.C;
    T *dst = gX0;
    if (np > 1) {
      chain_part_.ensure((size_t) np * stride * sizeof(T));
      dst = chain_part_.as<T>();
    }
    std::vector<void *> args = {&X0, &X1, &P21, &P22, &g2, &g3, &g4, &g21, &dst, &W, &nat, &one};
    if (np > 1) {
      args.push_back(&stride);
      for (unsigned long long &m : ck.parts[np].mask) args.push_back(&m);
    }
    HIP_CHECK(hipModuleLaunchKernel(np > 1 ? ck.bwd_part : ck.bwd, blocks, np, 1, 256, 1, 1, 0, stream_, args.data(), nullptr));
    cur_flops_ += ck.flops_per_atom * n;
    return np;
  }
  template<class T, class K> void launch_chain_sum(K &ck, int n, int np, T *gX0)
  {
    const long long rows = (n + ck.atoms_per_block - 1) / ck.atoms_per_block * ck.atoms_per_block, row = (long long) ck.nf0 * ck.C, total = n * row;
    hipLaunchKernelGGL(k_chain_sum<T>, dim3((unsigned) ((total + 255) / 256)), dim3(256), 0, stream_, (const T *) chain_part_.as<T>(), rows * row, np,
                       ck.keep0, ck.nf0, ck.C, total, gX0);
  }
  DevBuf chain_part_;

  // ---- element-dependent reduces ------------------------------------------------------------------------------
  // The forward of a set: results to out0 (fp64 rows) and out1 (rows of T).  Few tiles: the functions of a reduce go to several
  // blocks, as long as those fill the chip no more than twice, and k_reduce_sum (5 us) adds their parts (128 atoms of GRACE-1L: 34
  // -> 11 us; the six reduces of GRACE-2L with 107 atoms: 69 -> 21 us in two sets; 251 tiles in two parts: 44 -> 41 us; 512 tiles:
  // 75 us whole, 74 + 5 in parts).  One part with ordered sums, whose bits must not follow the number of tiles.
  template<class T> void launch_reduce_fwd(DevReduces<T> &R, int ka, int kf, const int *mu, const T *X0, const T *X1, const T *X2, const T *X3, double *out0,
                                           T *out1, const int *tiles, int ntiles)
  {
    if (ntiles == 0) return;
    for (size_t first = 0; first < R.d.size(); first += kReduceSet) {
      const int nr = (int) std::min<size_t>(kReduceSet, R.d.size() - first);
      ReduceSet<T> set{};
      std::copy(R.d.begin() + first, R.d.begin() + first + nr, set.r);
      const int most = std::max(1, (R.max_jobs + kReduceWaves - 1) / kReduceWaves);
      const int parts = ordered_ ? 1 : std::max(1, std::min(most, 2 * ncu_ / (nr * ntiles)));
      if (parts > 1) red_part_.ensure((size_t) nr * ntiles * parts * 16 * 32 * sizeof(double));
#define GR_RED(KA, KF)                                                                                                                      \
  hipLaunchKernelGGL((k_reduce_fwd<T, KA, KF>), dim3(ntiles, nr, parts), dim3(64 * kReduceWaves), 0, stream_, set, mu, tiles, X0, X1, X2, X3, out0, out1, \
                     parts, red_part_.as<double>())
      switch (ka * 10 + kf) {
        case 11: GR_RED(1, 1); break; case 12: GR_RED(1, 2); break; case 14: GR_RED(1, 4); break;
        case 21: GR_RED(2, 1); break; case 22: GR_RED(2, 2); break; case 24: GR_RED(2, 4); break;
        case 41: GR_RED(4, 1); break; case 42: GR_RED(4, 2); break; case 44: GR_RED(4, 4); break;
        default: throw Error("unsupported channel widths");
      }
#undef GR_RED
      if (parts > 1)
        hipLaunchKernelGGL(k_reduce_sum<T>, dim3(ntiles, nr), dim3(512), 0, stream_, set, tiles, (const double *) red_part_.as<double>(), parts, out0, out1);
    }
  }
  // The reverse of a set, rows of `list`: added to the adjoints, or (overwrite) written.  Tiles of a wave: as many as leave
  // 16 waves per SIMD to deal out, eight at most.  As a launch per reduce with a wave per row and tile, added to cleared rows:
  // GRACE-2L with 32 000 atoms 0.96 ms in 12 launches + 0.29 ms of fills, now 0.46 ms in two; 107 atoms 106 -> 14 us; GRACE-1L, one
  // reduce: 8192 atoms 75 -> 55 us, 65 536 in fp32 470 -> 305 (389 with a tile per wave, 310 with 4 or 16 for all).
  template<class T> void launch_reduce_bwd(DevReduces<T> &R, std::vector<std::unique_ptr<typename DevReduces<T>::List>> &list, const int *mu, const double *g0,
                                           const T *g1, T *G0, T *G1, T *G2, T *G3, const int *tiles, int ntiles, bool overwrite)
  {
    for (size_t q = 0; q < list.size(); q++) {
      const int njobs = (int) list[q]->host.size();
      if (njobs == 0 || ntiles == 0) continue;
      const int tpw = std::max(1, std::min(8, (int) ((long long) njobs * ntiles / (64 * ncu_))));
      hipLaunchKernelGGL(k_reduce_bwd<T>, dim3(njobs, (ntiles + 4 * tpw - 1) / (4 * tpw)), dim3(256), 0, stream_, list[q]->dev.template as<ReduceBwdJob>(),
                         R.WB.template as<T>(), R.drow, mu, tiles, ntiles, tpw, g0, g1, G0, G1, G2, G3, overwrite && q == 0 ? 1 : 0);
    }
  }
  DevBuf red_part_;

  // ---- exchange with ghost atoms ------------------------------------------------------------------------------
  void exchange_forward(int layer)
  {
    if (!exchange_.forward || n_nodes_ == n_) return;
    HIP_CHECK(hipStreamSynchronize(stream_));
    exchange_.forward(exchange_.user, layer);
  }
  void exchange_reverse(int layer)
  {
    if (!exchange_.reverse || n_nodes_ == n_) return;
    HIP_CHECK(hipStreamSynchronize(stream_));
    exchange_.reverse(exchange_.user, layer);
  }
  // The four row movers on rows [atom][function][CP] of which the first nf functions and C channels travel
  // (nf C doubles per atom); stride: elements per atom.
  template<class T> void move_rows(int mode, T *rows, long long stride, int nf, int C, int CP, int n, const int *list, int first, double *buf, bool host)
  {
    HIP_CHECK(hipSetDevice(device_));
    if (n <= 0) return;
    if (!rows) throw Error(who_ + ": the message rows do not exist yet (the exchange runs inside a pass)");
    const bool by_list = mode == 0 || mode == 3;
    if (by_list && !list) throw InvalidArgument("the atom list of the exchange is missing");
    if (!buf) throw InvalidArgument("the buffer of the exchange is missing");
    const size_t count = (size_t) n * nf * C;
    const int *dl = list;
    double *db = buf;
    if (host) {
      comm_buf_.ensure(count * sizeof(double));
      db = comm_buf_.as<double>();
      if (by_list) {
        for (int k = 0; k < n; k++)
          if (list[k] < 0 || list[k] >= n_nodes_) throw InvalidArgument("the atom list of the exchange names an atom outside the owned and ghost atoms");
        comm_list_.ensure((size_t) n * sizeof(int));
        HIP_CHECK(hipMemcpyAsync(comm_list_.p, list, (size_t) n * sizeof(int), hipMemcpyHostToDevice, stream_));
        dl = comm_list_.as<int>();
      }
      if (mode == 1 || mode == 3) HIP_CHECK(hipMemcpyAsync(db, buf, count * sizeof(double), hipMemcpyHostToDevice, stream_));
    }
    if (!by_list && (first < 0 || first + n > n_nodes_)) throw InvalidArgument("the atom range of the exchange lies outside the owned and ghost atoms");
    const size_t moved = mode == 1 ? (size_t) n * nf * CP : count;    // rows that are set are set with their padding
    const dim3 grid((unsigned) ((moved + 255) / 256)), block(256);
    if (mode == 0 || mode == 2)
      hipLaunchKernelGGL(k_comm_pack<T>, grid, block, 0, stream_, (const T *) rows, stride, nf, C, CP, by_list ? dl : nullptr, first, n, db);
    else
      hipLaunchKernelGGL((mode == 3 ? k_comm_unpack<T, true> : k_comm_unpack<T, false>), grid, block, 0, stream_, rows, stride, nf, C, CP,
                         by_list ? dl : nullptr, first, n, (const double *) db);
    HIP_CHECK(hipGetLastError());
    if (host && (mode == 0 || mode == 2)) HIP_CHECK(hipMemcpyAsync(buf, db, count * sizeof(double), hipMemcpyDeviceToHost, stream_));
    HIP_CHECK(hipStreamSynchronize(stream_));
  }

  // ---- one radial row for both directions of a bond (k_edge_pairs) ----
  // want_pairs_: set by an engine before begin_pass(), from pair_rows_min() bonds of the list on.  Measured: GRACE-1L with
  // 475 136 bonds, network 0.548 -> 0.281 ms, search 0.035 ms; GRACE-2L with 2.5 M bonds, both networks 6.0 -> 2.76 ms, search
  // 0.16 ms, of the kernels that gather the rows k_pair_fwd (then through LDS) 1.40 -> 1.64 ms and the others as before.  Not with tables, where
  // a row costs its stores only (312 018 bonds: 0.080 -> 0.047 ms, less than the search and the gathers).  Not from 2^31 listed
  // bonds on: the numbers of rows are 32-bit integers (begin_pass).
  // The search of a short list takes some 20 us whatever the list, and a network that has few tiles of 16 rows for each SIMD
  // does not get quicker by half when half of them go.  The line is at three tiles per SIMD of listed bonds and one network in
  // fp64, where a tile takes twice as long as in fp32; two networks share one search.  A call with own rows over one with
  // shared rows, fp64 / fp32: GRACE-1L, 33 560 bonds 0.992 / 0.949, 50 614 1.000 / 0.958, 74 082 1.075 / 0.995, 127 892 1.115 /
  // 1.034; GRACE-2L, 13 568 bonds 0.953 / 0.954, 25 046 1.002 / 0.968, 43 368 1.020 / 0.967, 59 080 1.033 / 1.014.  (Listed
  // bonds: how many lie inside the cutoff is known on the device only.)
  // GRACE_HIP_PAIR_ROWS=n: from n bonds on.
  int64_t pair_rows_min(int networks, size_t value_bytes) const
  {
    if (pair_rows_from_ >= 0) return pair_rows_from_;
    return (value_bytes == 8 ? 3 : 6) * (int64_t) 4 * ncu_ * 16 / networks;
  }
  int64_t pair_rows_from_ = pair_rows_switch();
  static int64_t pair_rows_switch()
  {
    const char *e = std::getenv("GRACE_HIP_PAIR_ROWS");
    return e && e[0] ? std::atoll(e) : -1;
  }
  DevBuf erow_, uid_, ux_, nrows_;
  static constexpr double kPairRowBytes = 2 * sizeof(int) + sizeof(double);    // erow_, uid_, ux_, per bond
  bool want_pairs_ = false, paired_ = false;
  int pair_chunks_ = 0;
  // chunks of cs atoms; bounds: first bond of every chunk (empty: one chunk of all atoms)
  void pair_rows(int cs, const std::vector<long long> &bounds)
  {
    paired_ = want_pairs_;
    if (!paired_) return;
    const int n = n_, nch = pair_chunks_ = (n + cs - 1) / cs;
    uid_.ensure((size_t) nb_ * sizeof(int));
    ux_.ensure((size_t) nb_ * sizeof(double));
    nrows_.ensure((size_t) nch * sizeof(long long));
    stage("edge_pairs", [&] {
      HIP_CHECK(hipMemsetAsync(nrows_.p, 0, (size_t) nch * sizeof(long long), stream_));
      for (int k = 0; k < nch; k++) {
        const int a0 = k * cs, nc = std::min(n, a0 + cs) - a0;
        const long long eb = bounds.empty() ? 0 : bounds[(size_t) k], ne = bounds.empty() ? nb_ : bounds[(size_t) k + 1] - eb;
        if (ne <= 0) continue;    // a chunk of isolated atoms
        hipLaunchKernelGGL(k_edge_pairs, dim3((unsigned) ((nc + 3) / 4)), dim3(256), 0, stream_, eoff_.as<long long>(), a0, nc, ej_.as<int>(),
                           rh_.as<double>(), xr_.as<double>(), erow_.as<int>(), ordered_ ? 0.0 : kSameArgument);
        hipLaunchKernelGGL(k_edge_rows, dim3((unsigned) ((ne + kRowsPerBlock - 1) / kRowsPerBlock)), dim3(1024), 0, stream_, eoff_.as<long long>(), a0,
                           nc, erow_.as<int>(), xr_.as<double>(), uid_.as<int>() + eb, ux_.as<double>() + eb, nrows_.as<unsigned long long>() + k);
      }
    });
  }
  PairedRows paired(int chunk, long long eb) const
  {
    PairedRows p;
    if (!paired_) return p;
    p.on = true;
    p.uid = uid_.as<int>() + eb;
    p.erow = erow_.as<int>();
    p.x = ux_.as<double>() + eb;
    p.n = nrows_.as<long long>() + chunk;
    return p;
  }

  // ---- chunks of atoms ---------------------------------------------------------------------------------------
  // Atoms per pass for a structure whose work buffers take `per_atom` bytes per atom of a chunk and `kept` bytes per atom
  // of the structure (without what pair_rows() keeps), after the reference's policy (libgrace/include/grace/kk/support.h:425-450): everything in one pass
  // while that fits 70 % of the memory this engine can have (the free device memory, or what the library's own cap
  // leaves, plus what its work buffers hold already), else the largest power of two >= 512 that fits.  Returns n for one pass.
  int plan_chunk(int n, double per_atom, double kept)
  {
    if (n <= 0 || chunk_request_ == 0) return n;
    if (chunk_request_ > 0) return std::min(n, chunk_request_);
    size_t free_b = 0, total_b = 0;
    HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    double avail = (double) free_b + (double) device_pool().held_on(device_);
    const long long cap = dev_bytes_limit().load();
    if (cap > 0) avail = std::min(avail, (double) (cap - dev_bytes_in_use().load()));
    double held = 0.0;
    for (const DevBuf *b : bufs_)
      if (!b->model_data) held += (double) b->bytes;
    const double budget = 0.7 * (avail + held);
    const double grown = 1.125;    // DevBuf::ensure
    kept += want_pairs_ ? kPairRowBytes * (double) nb_ / n : 0.0;
    if (grown * (per_atom * n + kept * n) <= budget) return n;
    int c = std::min(n, kChunkFloor);
    while (2 * c < n && grown * (per_atom * 2.0 * c + kept * n) <= budget) c *= 2;
    log_message(0, who_ + ": chunksize auto: " + std::to_string(c) + " atoms per pass for " + std::to_string(n) + " atoms (" +
                       std::to_string((long long) (per_atom * 1000 / 1048576)) + " MB of work buffers and " +
                       std::to_string((long long) (kept * 1000 / 1048576)) + " MB kept per 1000 atoms, " + std::to_string((long long) (avail / 1048576)) +
                       " MB of device memory available)");
    return c;
  }
  static constexpr int kChunkFloor = 512;    // smallest chunk of the automatic choice and of the retries after a failed allocation
  // Tiles of 16 atoms of one element for every chunk of `cs` atoms, with atom indices counted from the chunk's first atom:
  // chunk k owns tiles [chunk_tile_off_[k], chunk_tile_off_[k + 1]) of chunk_tiles_.
  void layout_chunks(int cs)
  {
    if (chunk_laid_out_ == cs) return;
    const int n = n_, nch = (n + cs - 1) / cs;
    std::vector<int> all, el;
    chunk_tile_off_.assign(1, 0);
    chunk_tile_el_.clear();
    for (int k = 0; k < nch; k++) {
      const int a0 = k * cs, a1 = std::min(n, a0 + cs);
      const std::vector<int> sub(mu_host_.begin() + a0, mu_host_.begin() + a1);
      const std::vector<int> t = element_tiles(sub, nelem_, el);
      all.insert(all.end(), t.begin(), t.end());
      chunk_tile_off_.push_back((int) all.size() / 16);
      chunk_tile_el_.push_back(el);    // tiles of element e within the chunk: [el[e], el[e + 1])
    }
    upload_vec(chunk_tiles_, all);
    chunk_laid_out_ = cs;
  }
  // first edge of every chunk (and the end of the last): eoff at the chunk boundaries, read back after the bond filter
  std::vector<long long> chunk_edge_bounds(int cs)
  {
    const int nch = (n_ + cs - 1) / cs;
    std::vector<long long> b((size_t) nch + 1);
    for (int k = 0; k <= nch; k++)
      HIP_CHECK(hipMemcpyAsync(&b[(size_t) k], eoff_.as<long long>() + std::min(n_, k * cs), sizeof(long long), hipMemcpyDeviceToHost, stream_));
    HIP_CHECK(hipStreamSynchronize(stream_));
    return b;
  }
  // a pointer moved back by `count` elements: kernels that index a chunk's buffer with structure-wide indices (edges)
  template<class U> static U *moved_back(U *p, long long count)
  {
    return reinterpret_cast<U *>(reinterpret_cast<intptr_t>(p) - (intptr_t) (count * (long long) sizeof(U)));
  }
  bool chunks_ = false;          // the engine can evaluate a structure in chunks of atoms
  int chunk_request_ = -1, chunk_used_ = 0, chunk_laid_out_ = 0;
  std::vector<int> mu_host_, chunk_tile_off_;
  std::vector<std::vector<int>> chunk_tile_el_;
  DevBuf chunk_tiles_;

  int device_, ncu_ = 256;
  std::string arch_, who_;
  int ntypes_;
  std::vector<int> type2mu_;
  int nelem_;
  std::vector<double> cut_host_;
  // uploaded structure
  int n_nodes_ = 0;           // central atoms and ghosts (= n_ without ghosts)
  uint64_t upload_serial_ = 0;
  PinnedBuf pin_in_, pin_out_;    // staging of the positions of a call and of what a call returns
  PinnedBuf pin_flag_;            // the zero-bond flag of the last pass (two ints)
  DevBuf vatom_;              // per-atom virials [n_nodes][9] (xx yy zz xy xz yz yx zx zy) of a pass with the vatom flag
  bool ran_vatom_ = false;
  double *vatom_ptr() { return ran_vatom_ ? vatom_.as<double>() : nullptr; }
  ExchangeCallbacks exchange_{};
  DevBuf comm_list_, comm_buf_;    // staging of the host forms of the row movers
  int n_ = 0, n_peak_ = 0;    // atoms of the uploaded structure; of the largest pass since the work buffers were released
  int64_t nb_ = 0;
  bool have_rij_ = false;
  DevBuf cut_, mu_, sid_, offset_, j_, rij_, x_, image_, shifts_, tiles_;
  int ntiles_ = 0, nstruct_ = 1;
  std::vector<int> tile_el_;    // [nel + 1] tile range of every element
  bool have_sid_ = false, sid_sorted_ = true;    // sid_sorted_: the atoms of every structure are one range of rows

  // ---- ordered sums (engines that set ordered_ok_): the reverse kernels store the force of every bond on its central atom
  // (fedge_[e][3]) and, per atom, the sums over its own bonds (fcen_[i][9]: force, then the six virial sums) instead of
  // adding with atomics; the forces on the neighbours are gathered through the bonds listed by neighbour atom (rebuilt every
  // pass: the bonds inside the cutoff change with the positions); energy and virial records are summed per structure in a
  // fixed order from the per-atom energies and fcen_
  bool ordered_ok_ = false, ordered_ = false;
  int spline_n_ = 0;
  // the engine's radial kernels take the setting (engines without radial tables say so and stay exact)
  virtual void apply_spline(int n)
  {
    if (n > 0) log_message(0, who_ + ": radial tables are not used by this engine; the radial MLPs are evaluated for every bond");
  }
  DevBuf fedge_, fcen_, tcount_, toff_, traw_, tsorted_;
  // before begin_pass(): what the mode cannot do
  void ordered_check(const RunFlags &fl) const
  {
    if (!ordered_) return;
    if (fl.vatom && !fl.energy_only) throw InvalidArgument(who_ + ": per-atom virials are not available with ordered sums");
    if (!sid_sorted_) throw InvalidArgument(who_ + ": ordered sums need the atoms of every structure in one range of rows");
    if (nb_ >= INT32_MAX) throw InvalidArgument(who_ + ": ordered sums number the bonds with 32 bits");
  }
  // after begin_pass() of a pass with forces: the per-bond and per-atom stores, and the bonds by neighbour atom, each row
  // in ascending order
  void ordered_begin()
  {
    const int n = n_, nn = n_nodes_;
    const size_t ne = (size_t) std::max<int64_t>(nb_, 1);
    fedge_.ensure(3 * ne * sizeof(double));
    fcen_.ensure((size_t) 9 * std::max(n, 1) * sizeof(double));
    tcount_.ensure((size_t) 2 * nn * sizeof(int));    // bonds per neighbour atom, then the fill cursors
    toff_.ensure(((size_t) nn + 1) * sizeof(long long));
    traw_.ensure(ne * sizeof(int));
    tsorted_.ensure(ne * sizeof(int));
    stage("ordered_list", [&] {
      HIP_CHECK(hipMemsetAsync(tcount_.p, 0, (size_t) 2 * nn * sizeof(int), stream_));
      const long long *n_edges = eoff_.as<long long>() + n;
      const dim3 egrid((unsigned) ((ne + 255) / 256)), agrid((unsigned) ((nn + 3) / 4));
      hipLaunchKernelGGL(k_tlist_count, egrid, dim3(256), 0, stream_, n_edges, ej_.as<int>(), tcount_.as<int>());
      launch_scan(stream_, tcount_.as<int>(), nn, toff_.as<long long>());
      hipLaunchKernelGGL(k_tlist_fill, egrid, dim3(256), 0, stream_, n_edges, ej_.as<int>(), toff_.as<long long>(), tcount_.as<int>() + nn,
                         traw_.as<int>());
      hipLaunchKernelGGL(k_tlist_sort, agrid, dim3(256), 0, stream_, nn, toff_.as<long long>(), traw_.as<int>(), tsorted_.as<int>());
    });
  }
  // end of the pass: forces of all rows (ghosts included) and the records of the structures
  void ordered_finish(const RunFlags &fl)
  {
    const int n = n_, nn = n_nodes_;
    stage("ordered_sums", [&] {
      if (!fl.energy_only)
        hipLaunchKernelGGL(k_ordered_forces, dim3((unsigned) ((nn + 3) / 4)), dim3(256), 0, stream_, nn, n, toff_.as<long long>(), tsorted_.as<int>(),
                           fedge_.as<double>(), fcen_.as<double>(), f_.as<double>());
      hipLaunchKernelGGL(k_ordered_records, dim3((unsigned) nstruct_), dim3(256), 0, stream_, n, sid_ptr(), eatom_.as<double>(), fcen_.as<double>(),
                         fl.energy_only ? 0 : 1, scal_.as<double>());
    });
  }
  const int *sid_ptr() const { return have_sid_ ? sid_.as<int>() : nullptr; }
  // records (energy, virial[6], unused) of the pass: one per structure of a list with structure indices, kRecordCopies of one
  // structure (record_of)
  int record_copies() const { return have_sid_ ? 1 : kRecordCopies; }
  size_t records() const { return (size_t) nstruct_ * record_copies(); }
  void add_records(const double *rec, int structure, double *sum) const
  {
    for (int k = 0; k < 7; k++) sum[k] = 0.0;
    for (int q = 0; q < record_copies(); q++)
      for (int k = 0; k < 7; k++) sum[k] += rec[8 * ((size_t) structure * record_copies() + q) + k];
  }
  // edges of the pass and its outputs (scal: energy, virial[6])
  DevBuf count_, eoff_, zero_, ei_, ej_, emu_, rh_, r_, xr_, rc_, eatom_;
  // records of the structures, then the forces, in one buffer that is cleared and fetched at once; laid out by begin_pass()
  struct View {
    double *p = nullptr;
    template<class U> U *as() const { static_assert(std::is_same<U, double>::value, "records and forces are fp64"); return p; }
  };
  DevBuf out_;
  View scal_, f_;
  bool ran_ = false, ran_forces_ = false, ran_eatom_ = false, ran_uq_ = false;
  bool has_uq_head_ = false;      // set by an engine whose model carries a valid UQ head
  std::string uq_why_ = "this engine evaluates none";
  DevBuf uq_gamma_, uq_sigma_, uq_cluster_;
  hipStream_t stream_ = nullptr;
  bool profile_ = false;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> events_;
  std::vector<std::string> ev_names_;
  std::vector<double> ev_flops_;
  double cur_flops_ = 0.0;
  size_t ev_used_ = 0;
  std::vector<StageTime> times_;
  // the reverse pair kernel on the matrix cores wherever it applies; GRACE_HIP_PAIR_MFMA=0: the vector kernels
  int pair_mfma_ = pair_mfma_switch();
  static int pair_mfma_switch()
  {
    const char *e = std::getenv("GRACE_HIP_PAIR_MFMA");
    return e && e[0] == '0' ? 0 : 1;
  }
  // the sums of the bonds that kernel leaves for k_bond_bwd of the first layer (BondBwdArgs::bsum): cleared once per pass
  DevBuf bsum_;
  bool bsum_on_ = false;
  double *bsum_ptr() const { return bsum_on_ ? bsum_.as<double>() : nullptr; }
  size_t bsum_bytes() const { return (size_t) 3 * std::max<int64_t>(nb_, 1) * sizeof(double); }
  void bsum_begin(bool on, bool clear = true)    // clear == false: the caller clears bsum_bytes() of them
  {
    bsum_on_ = on;
    if (!on) return;
    const size_t bytes = bsum_bytes();
    bsum_.ensure(bytes);
    if (clear) stage("zero_bond_sums", [&] { HIP_CHECK(hipMemsetAsync(bsum_.p, 0, bytes, stream_)); });
  }
  int pair_waves_ = pair_waves_switch();    // waves of a block of that kernel; 0: those of one group of slots
  static int pair_waves_switch()
  {
    const char *e = std::getenv("GRACE_HIP_PAIR_WAVES");
    const int w = e ? std::atoi(e) : 0;
    return w >= 1 && w <= 8 ? w : 0;
  }
  int drow_[16];
  int drow64_[16];    // fp32 engines: the accumulator rows of the fp64 MFMA (the fp64 radial MLP that fills the radial tables)
  // probes the MFMA accumulator layout of the engine's precision; an fp32 engine probes the fp64 one first and keeps it
  template<class T> void probe_mfma_both()
  {
    if constexpr (sizeof(T) == 4) {
      probe_mfma<double>();
      for (int q = 0; q < 16; q++) drow64_[q] = drow_[q];
    }
    probe_mfma<T>();
    if constexpr (sizeof(T) == 8)
      for (int q = 0; q < 16; q++) drow64_[q] = drow_[q];
  }
};

}    // namespace grhip
