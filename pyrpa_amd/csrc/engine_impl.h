// Convolution engine (see engine.h): the member templates, instantiated per
// precision in engine_f64.hip and engine_f32.hip.
//
// Restructure relative to the reference (same mathematics):
//  * The reference transforms two full grids per orbital pair and per call
//    (fchi.f90:584-585, fself.f90:239-240).  Here every full-grid G_ab is
//    transformed once (No^2 FFTs) and reused by all chi pairs and by Sigma.
//  * Sigma accumulates V*G products per output (m1,l1) in (r,tau) space
//    before one inverse FFT, instead of one inverse FFT per vertex pair
//    (fself.f90:257): No^2 instead of Nchi^2 inverse transforms.
//  * The tail correction conv[G] - conv[G0] + ref[G0] (fchi.f90:852-892) is
//    combined in (r,tau) space before a single inverse FFT per pair.
#pragma once
#include <cmath>
#include <cstdlib>

#include <array>
#include <map>

#include "engine.h"

namespace gmod {

constexpr double PI_E = 3.141592653589793238462643383279;

static bool sigma_unfused() {
  const char* e = getenv("GMOD_SIGMA_UNFUSED");
  return e && *e && *e != '0';
}
// GMOD_SIGMA_UNGROUPED=1: the Sigma increment's accumulating pass reads the
// three operands of every source instead of the grouped form
static bool sigma_ungrouped() {
  const char* e = getenv("GMOD_SIGMA_UNGROUPED");
  return e && *e && *e != '0';
}
// GMOD_SIGMA_ACCUM=1: the Sigma increment in the grouped accumulating-pass
// form instead of the contraction form
static bool sigma_accum_form() {
  const char* e = getenv("GMOD_SIGMA_ACCUM");
  return e && *e && *e != '0';
}

template <typename R>
ConvEngine<R>::ConvEngine(const Mesh& m, const OrbPairs& p) : mesh(m), op(p) {
  N = m.N();
  p4 = &fft_plan<R>(m.Nx, m.Ny, m.Nz, m.M, 15);
  p3 = &fft_plan<R>(m.Nx, m.Ny, m.Nz, m.M, 7);
  work.alloc(N);
  tmp.alloc(N);
  rhobar.alloc((size_t)p.No * p.No);
  ol_h.resize(2 * (size_t)p.Nchi);
  for (int l = 0; l < p.Nchi; ++l) {
    ol_h[2 * l] = p.ol[l][0];
    ol_h[2 * l + 1] = p.ol[l][1];
  }
  ol_d.alloc(ol_h.size());
  ol_d.upload(ol_h.data(), ol_h.size(), ctx().stream);
  if (p.soc) {
    soc_inv.set(std::vector<int>(p.inv.begin(), p.inv.end()), ctx().stream);
    soc_spin.set(p.spin, ctx().stream);
  }
  // the tables of the computed pairs: all of them, and apart those that are
  // their own partner (the tail conjugates their sum half way)
  auto table = [&](PairTab& t, int which, bool partners) {  // 0 all, 1 self-partner, 2 the others
    std::vector<int> pr, ga;
    for (auto& lm : p.irr) {
      const int l = lm[0], mm = lm[1];
      const auto q = p.partner[mm + p.Nchi * l];
      const bool self = q[0] == mm && q[1] == l;
      if ((which == 1 && !self) || (which == 2 && self)) continue;
      pr.push_back(p.ol[l][0] + p.No * p.ol[mm][0]);
      pr.push_back(p.ol[mm][1] + p.No * p.ol[l][1]);
      ga.push_back(mm + p.Nchi * l);
      ga.push_back(partners && q[0] >= 0 ? q[0] + p.Nchi * q[1] : -1);
      ga.push_back(l + p.Nchi * mm);
      ga.push_back((which == 1 ? 1 : 0) + (p.psign[mm + p.Nchi * l] < 0 ? 2 : 0));
    }
    t.n = (int)pr.size() / 2;
    t.prod.set(std::move(pr), ctx().stream);
    t.gat.set(std::move(ga), ctx().stream);
  };
  table(pairs_all, 0, true);
  table(pairs_self, 1, false);
  table(pairs_other, 2, true);
  // without the conjugation and the partner: the second sum of a self-partner
  // pair, and the plain store of every pair
  auto plain = [&](const PairTab& from, PairTab& to) {
    to.n = from.n;
    to.prod.set(from.prod.h, ctx().stream);
    std::vector<int> ga = from.gat.h;
    for (int i = 0; i < to.n; ++i) {
      ga[4 * i + 1] = -1;
      ga[4 * i + 3] = 0;
    }
    to.gat.set(std::move(ga), ctx().stream);
  };
  plain(pairs_self, self_plain);
  plain(pairs_all, all_plain);
  plain(pairs_other, other_plain);
  std::vector<int> ga;
  for (int o = 0; o < p.No * p.No; ++o) {
    const int e[4] = {o, -1, 0, 0};
    ga.insert(ga.end(), e, e + 4);
  }
  orb_gat.set(std::move(ga), ctx().stream);
}

template <typename R>
void ConvEngine<R>::fft(cpx<R>* g, int sign, bool spatial_only, hipStream_t s) {
  const FFTPlan<R>* p = spatial_only ? p3 : p4;
  R sc = sign > 0 ? (R)(1.0 / (double)p->transformed_points()) : (R)1;
  p->exec(g, tmp.p, sign, sc, s);
}

template <typename R>
void ConvEngine<R>::transform_green(const zd* G, bool g0, hipStream_t s) {
  DBuf<cpx<R>>& dst = g0 ? F0g : Fg;
  const int No = op.No;
  if (dst.n != (size_t)(No * No) * N) dst.alloc((size_t)No * No * N);
  const MeshDev md = mesh_dev(mesh);
  const GridStore<R> gs{dst.p, (unsigned)mesh.Nkall, N};
  if (op.soc)
    p4->exec_batch(SocGreenBatch<R>{G, No, soc_inv.ptr(), soc_spin.ptr(), md}, gs, dst.p, No * No, tmp.p, -1, (R)1, s);
  else
    p4->exec_batch(GreenBatch<R>{G, No, md}, gs, dst.p, No * No, tmp.p, -1, (R)1, s);
}

template <typename R>
cpx<R>* ConvEngine<R>::work_grids(int n) {
  if (work.n < (size_t)n * N) work.alloc((size_t)n * N);
  return work.p;
}

// n inverse transforms of products (PL: a batch of ProductLoad or
// IncProductLoad), item i gathered by item i of gat, in batches
template <typename R>
template <class PL>
void ConvEngine<R>::product_batches(const PL& pl, const GatherBatch<R>& gat, int n, hipStream_t s) {
  const R invN = (R)(1.0 / (double)p4->transformed_points());
  const int step = p4->batch_items(n);
  for (int i0 = 0; i0 < n; i0 += step) {
    const int m = std::min(step, n - i0);
    p4->exec_batch(pl.from(i0), gat.from(i0), work_grids(std::min(step, n)), m, tmp.p, +1, invN, s, true);
  }
}

// TA, TB of every orbital pair written out by an elementwise kernel (the
// exponentials advance by a factor per slot, at full occupancy) and then
// transformed; above 8 orbitals the functions are evaluated inside the
// transform's first pass instead
template <typename R>
void ConvEngine<R>::tau_grids(cpx<R>* ta, cpx<R>* tb, const double* eig_d, const zd* uni_d, double mu, double mu2,
                              bool diff, double temp, hipStream_t s) {
  const int No = op.No;
  const double beta = 1.0 / temp, dtau = beta / (double)mesh.M;
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  if (No <= 8) {
    tau_ref_grids<R>(ta, tb, eig_d, uni_d, No, mu, mu2, diff, beta, dtau, md, s);
    p3->exec_many(ta, No * No, tmp.p, -1, (R)1, s);
    p3->exec_many(tb, No * No, tmp.p, -1, (R)1, s);
    return;
  }
  for (int ab = 0; ab < No * No; ++ab)
    for (int which = 0; which < 2; ++which) {
      const int a = ab % No, b = ab / No;
      cpx<R>* t = (which == 0 ? ta : tb) + (long)ab * N;
      if (diff) {
        const TauRefLoad<double> cur{eig_d, uni_d, a, b, No, which, mu, beta, dtau, md};
        const TauRefLoad<double> prev{eig_d, uni_d, a, b, No, which, mu2, beta, dtau, md};
        p3->exec_fused(TauRefDiffLoad<R>{cur, prev}, GridStore<R>{t, S}, t, tmp.p, -1, (R)1, s);
      } else {
        p3->exec_fused(TauRefLoad<R>{eig_d, uni_d, a, b, No, which, mu, beta, dtau, md}, GridStore<R>{t, S}, t, tmp.p,
                       -1, (R)1, s);
      }
    }
}

// Tail constants of chi0 at chemical potential mu (fchi.f90:731-772):
// J[l + Nchi*m] = delta_{a13 b13} rhobar_{a42 b42} - delta_{a42 b42} rhobar_{a13 b13}
// with rhobar the BZ-averaged free density matrix, and the sawtooth correction
// sawc(nu_j) of the discrete tau reference; both stay on the device.
template <typename R>
void ConvEngine<R>::tail_constants(double temp, const double* eig_d, const zd* uni_d, double mu, DBuf<zd>& J,
                                   DBuf<zd>& sawc_d, hipStream_t s) const {
  const int No = op.No, Nchi = op.Nchi;
  if (J.n != (size_t)Nchi * Nchi) J.alloc((size_t)Nchi * Nchi);
  tail_density(rhobar.p, eig_d, uni_d, No, mu, 1.0 / temp, mesh_dev(mesh), s);
  tail_jumps(J.p, rhobar.p, ol_d.p, No, Nchi, s);
  if (sawc_d.n == (size_t)mesh.Nw) return;
  sawc_d.alloc(mesh.Nw);
  sawtooth(sawc_d.p, mesh.Nw, temp, s);
}

template <typename R>
GatherStore<R> ConvEngine<R>::gather_sf(zd* dst, double w, const zd* J, const zd* sawc, int acc, hipStream_t s) {
  if (!tlive_built) {
    for (int small = 0; small < 2; ++small) {
      const std::vector<unsigned char> h = p4->fwd_last_live(mesh.kgat_host, &tlive_frac[small], small != 0);
      if (h.empty()) continue;
      tlive[small].alloc(h.size());
      tlive[small].upload(h.data(), h.size(), s);
      GMOD_HIP(hipStreamSynchronize(s));  // h is released here
    }
    tlive_built = true;
  }
  GatherStore<R> g{dst, w, J, sawc, acc, mesh_dev(mesh)};
  if (tlive[0].n) {
    g.live = tlive[0].p;
    g.live_frac = tlive_frac[0];
  }
  if (tlive[1].n) {
    g.live_s = tlive[1].p;
    g.live_s_frac = tlive_frac[1];
  }
  return g;
}

template <typename R>
void ConvEngine<R>::chi0(zd* chi, double temp, bool tail, const double* eig_d, const zd* uni_d, double mu,
                         hipStream_t s, bool apply_threshold) {
  const int No = op.No, Nchi = op.Nchi;
  const long NkNw = mesh.Nk * (long)mesh.Nw;
  const double w = temp / (double)mesh.Nkall;
  if (tail && sizeof(R) < sizeof(double)) {
    // the tail subtraction stays FP64 when the transforms are FP32
    chi0_split_tail(chi, temp, eig_d, uni_d, mu, s);
    if (apply_threshold) threshold(chi, NkNw * Nchi * Nchi, 1e-9, s);
    return;
  }
  const MeshDev md = mesh_dev(mesh);
  if (!mesh.complete) GMOD_HIP(hipMemsetAsync(chi, 0, NkNw * Nchi * Nchi * sizeof(zd), s));
  // the partner copies are written by the gather on a complete mesh (every
  // slot of a slice is written), else apart
  const bool fuse = mesh.complete;
  auto gather = [&](const PairTab& t, double wt, const zd* J, const zd* saw, int acc) {
    return GatherBatch<R>{chi, NkNw, t.gat.ptr(), gather_sf(chi, wt, J, saw, acc, s)};
  };
  if (!tail) {
    // every product is G13(r,t) G42(-r,-t): the mirrored G grids are formed
    // once (coalesced) and then read in place.  The inverse transforms run
    // spatial-first, so a (-r,-t) operand that is not mirrored (the tail
    // terms) is read as whole reversed planes.
    if (Mg.n != Fg.n) Mg.alloc(Fg.n);
    mirror_grid(Mg.p, Fg.p, mesh.Nx, mesh.Ny, mesh.Nz, mesh.M, No * No, s);
    const PairTab& t = fuse ? pairs_all : all_plain;
    product_batches(ProductBatch<R, 1>{{Fg.p}, {Mg.p}, {(R)-1}, {1}, N, t.prod.ptr(), md, 1},
                    gather(t, w, nullptr, nullptr, 0), t.n, s);
    if (!fuse) partner_copies(chi, pairs_all.gat.d.p, pairs_all.n, NkNw, s);
  } else {
    DBuf<zd> Jt, sawc_d;
    {
      DBuf<zd> G0((size_t)NkNw * No * No);  // its block may be reused in stream order
      green0(G0.p, eig_d, uni_d, mu, temp, mesh.Nk, (int)mesh.Nw, No, s);
      transform_green(G0.p, true, s);
    }
    if (TA.n != (size_t)(No * No) * N) { TA.alloc((size_t)No * No * N); TB.alloc((size_t)No * No * N); }
    tau_grids(TA.p, TB.p, eig_d, uni_d, mu, mu, false, temp, s);
    tail_constants(temp, eig_d, uni_d, mu, Jt, sawc_d, s);
    const R wr = (R)(-1.0 / (temp * (double)mesh.Nkall));
    // conv[G] - conv[G0] + ref in one product
    const PairTab& t = fuse ? pairs_other : other_plain;
    product_batches(ProductBatch<R, 3>{{Fg.p, F0g.p, TA.p}, {Fg.p, F0g.p, TB.p}, {(R)(-w), (R)w, wr}, {1, 1, 0}, N,
                                       t.prod.ptr(), md},
                    gather(t, 1.0, Jt.p, sawc_d.p, 0), t.n, s);
    if (!fuse) partner_copies(chi, pairs_other.gat.d.p, pairs_other.n, NkNw, s);
    // A self-partner slice (partner == itself) is conjugated in place after each
    // of the reference's three accumulation passes (fchi.f90:610, 846); the net
    // result is conj(conv[G] + ref) - conv[G0].  It equals conj of the plain sum
    // whenever TRS holds; keep the reference's order so results match it on any
    // input.
    product_batches(ProductBatch<R, 2>{{Fg.p, TA.p}, {Fg.p, TB.p}, {(R)(-w), wr}, {1, 0}, N, pairs_self.prod.ptr(), md},
                    gather(pairs_self, 1.0, Jt.p, sawc_d.p, 0), pairs_self.n, s);
    product_batches(ProductBatch<R, 1>{{F0g.p}, {F0g.p}, {(R)w}, {1}, N, self_plain.prod.ptr(), md},
                    gather(self_plain, 1.0, nullptr, nullptr, 1), self_plain.n, s);
  }
  if (apply_threshold) threshold(chi, NkNw * Nchi * Nchi, 1e-9, s);
}

template <typename R>
void ConvEngine<R>::chi0_ff(zd* chi, const zd* F, const double* prt, bool singlet, double temp, hipStream_t s) {
  const int No = op.No, Nchi = op.Nchi;
  const long NkNw = mesh.Nk * (long)mesh.Nw;
  const double w = temp / (double)mesh.Nkall;
  // F(-k) = sgn F^T(k) and the gap's frequency parity dprt: both +1 for a
  // singlet, -1 for a triplet (ffeliash.f90:541-547)
  const double sgn = singlet ? 1.0 : -1.0, dprt = sgn;
  if (Lff.n != (size_t)2 * N) Lff.alloc((size_t)2 * N);
  cpx<R>* A = Lff.p;
  cpx<R>* B = Lff.p + N;
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  auto off = [&](int a, int b) { return NkNw * (long)(a + No * b); };
  if (!mesh.complete) GMOD_HIP(hipMemsetAsync(chi, 0, NkNw * Nchi * Nchi * sizeof(zd), s));
  for (auto& lm : op.irr) {
    const int l = lm[0], m = lm[1];
    const int l1 = op.ol[l][0], l2 = op.ol[l][1], m1 = op.ol[m][0], m2 = op.ol[m][1];
    const FFLoad<R> f14{F, off(m2, l1), off(l1, m2), off(m1, l1), off(l1, m2), prt[l1] * prt[m2] * sgn * dprt, 1, md};
    const FFLoad<R> f23{F, off(l2, m1), off(m1, l2), off(l2, m2), off(l2, m1), prt[m1] * prt[l2] * sgn * dprt, 0, md};
    p4->exec_fused(f14, GridStore<R>{A, S}, A, tmp.p, -1, (R)1, s);
    p4->exec_fused(f23, GridStore<R>{B, S}, B, tmp.p, -1, (R)1, s);
    ProductLoad<R> pl{};
    pl.m = md;
    pl.add(A, B, (R)-1, 1);
    zd* dst = chi + NkNw * (m + (long)Nchi * l);
    p4->exec_fused(pl.template fixed<1>(), gather_sf(dst, w, nullptr, nullptr, 0, s), work.p, tmp.p, +1,
                   (R)(1.0 / (double)p4->transformed_points()), s, true);
    auto pr = op.partner[m + Nchi * l];
    if (pr[0] >= 0) conj_copy(chi + NkNw * (pr[0] + (long)Nchi * pr[1]), dst, NkNw, s);
  }
  threshold(chi, NkNw * Nchi * Nchi, 1e-9, s);
}

template <typename R>
void ConvEngine<R>::tau_reference(zd* chi, double temp, const double* eig_d, const zd* uni_d, double mu,
                                  const zd* J, const zd* sawc_d, hipStream_t s) {
  const int No = op.No;
  const long NkNw = mesh.Nk * (long)mesh.Nw;
  if (TA.n != (size_t)(No * No) * N) { TA.alloc((size_t)No * No * N); TB.alloc((size_t)No * No * N); }
  tau_grids(TA.p, TB.p, eig_d, uni_d, mu, mu, false, temp, s);
  const double wref = 1.0 / (temp * (double)mesh.Nkall);
  product_batches(ProductBatch<R, 1>{{TA.p}, {TB.p}, {(R)(-wref)}, {0}, N, all_plain.prod.ptr(), mesh_dev(mesh)},
                  GatherBatch<R>{chi, NkNw, all_plain.gat.ptr(), gather_sf(chi, 1.0, J, sawc_d, 1, s)}, all_plain.n, s);
}

template <typename R>
void ConvEngine<R>::chi0_split_tail(zd* chi, double temp, const double* eig_d, const zd* uni_d, double mu,
                                    hipStream_t s) {
  const int No = op.No, Nchi = op.Nchi;
  const long Nk = mesh.Nk, Nw = mesh.Nw, NkNw = Nk * Nw;
  const double w = temp / (double)mesh.Nkall;
  {
    DBuf<zd> G0((size_t)NkNw * No * No);
    green0(G0.p, eig_d, uni_d, mu, temp, Nk, (int)Nw, No, s);
    transform_green(G0.p, true, s);
    GMOD_HIP(hipStreamSynchronize(s));  // G0 is released at the end of the scope
  }
  DBuf<zd> J, sawc_d;
  tail_constants(temp, eig_d, uni_d, mu, J, sawc_d, s);
  const MeshDev md = mesh_dev(mesh);
  if (!mesh.complete) GMOD_HIP(hipMemsetAsync(chi, 0, NkNw * Nchi * Nchi * sizeof(zd), s));
  auto gather = [&](const PairTab& t, int acc) {
    return GatherBatch<R>{chi, NkNw, t.gat.ptr(), gather_sf(chi, 1.0, nullptr, nullptr, acc, s)};
  };
  // 1) -w conv[G] + w conv[G0] at grid precision (a self-partner pair: -w conv[G] only)
  product_batches(ProductBatch<R, 2>{{Fg.p, F0g.p}, {Fg.p, F0g.p}, {(R)(-w), (R)w}, {1, 1}, N, other_plain.prod.ptr(), md},
                  gather(other_plain, 0), other_plain.n, s);
  product_batches(ProductBatch<R, 1>{{Fg.p}, {Fg.p}, {(R)(-w)}, {1}, N, self_plain.prod.ptr(), md},
                  gather(self_plain, 0), self_plain.n, s);
  // 2) + the tau reference and the sawtooth term, FP64
  {
    ConvEngine<double> e64(mesh, op);
    e64.tau_reference(chi, temp, eig_d, uni_d, mu, J.p, sawc_d.p, s);
    GMOD_HIP(hipStreamSynchronize(s));  // e64's grids are released at the end of the scope
  }
  // 3) the reference's order for a self-partner pair, conj(conv[G] + ref) -
  //    conv[G0] (fchi.f90:610, 846, 886); partner copies of the others
  for (int i = 0; i < pairs_self.n; ++i) {
    zd* dst = chi + NkNw * pairs_self.gat.h[4 * i];
    conj_copy(dst, dst, NkNw, s);
  }
  product_batches(ProductBatch<R, 1>{{F0g.p}, {F0g.p}, {(R)w}, {1}, N, self_plain.prod.ptr(), md},
                  gather(self_plain, 1), self_plain.n, s);
  partner_copies(chi, pairs_other.gat.d.p, pairs_other.n, NkNw, s);
}

template <typename R>
bool ConvEngine<R>::grouped_table(std::vector<int>& ytab) const {
  const int No = op.No, Nchi = op.Nchi, NAB = No * No;
  ytab.assign((size_t)NAB * NAB, -1);
  for (int l = 0; l < Nchi; ++l)
    for (int m = 0; m < Nchi; ++m) {
      const int o = op.ol[m][0] + No * op.ol[l][0], ab = op.ol[m][1] + No * op.ol[l][1];
      int& slot = ytab[(size_t)o * NAB + ab];
      if (slot >= 0) return false;
      slot = m + Nchi * l;
    }
  for (int v : ytab)
    if (v < 0) return false;
  return true;
}

template <typename R>
std::vector<std::array<int, 2>> ConvEngine<R>::share_heads(std::vector<int>& entry) const {
  const int Nchi = op.Nchi;
  std::vector<std::array<int, 2>> heads;
  entry.assign((size_t)Nchi * Nchi, -1);
  for (int l = 0; l < Nchi; ++l)
    for (int m = 0; m < Nchi; ++m) {
      const int t = l + Nchi * m;  // the transposed pair
      if (entry[t] >= 0) {
        entry[m + Nchi * l] = (entry[t] & ~1) + 1;
      } else {
        entry[m + Nchi * l] = 2 * (int)heads.size();
        heads.push_back({m, l});
      }
    }
  return heads;
}

template <typename R>
void ConvEngine<R>::head_offsets(std::vector<long>& offs, int m, int l) const {
  const long NC = mesh.Nk * (long)mesh.Nw;
  offs.push_back(NC * (m + (long)op.Nchi * l));
  offs.push_back(NC * (l + (long)op.Nchi * m));
}

template <typename R>
template <typename Sv>
void ConvEngine<R>::slot0_corr(cpx<R>* dh, const cpx<Sv>* V, const long* offs_d, int nh, hipStream_t s) {
  if (nh <= 0) return;
  const unsigned S = (unsigned)mesh.Nkall;
  const size_t n = (size_t)nh * S;
  if (dh_tmp.n < n) dh_tmp.alloc(n);
  const MeshDev md = mesh_dev(mesh);
  const unsigned grid = (unsigned)std::min<long>(((long)n + 255) / 256, 256L * 64);
  hipLaunchKernelGGL((k_slot0_diff<R, Sv>), dim3(grid), dim3(256), 0, s, dh, V, offs_d, nh, S, md);
  GMOD_CHECK_LAUNCH();
  fft_plan<R>(mesh.Nx, mesh.Ny, mesh.Nz, nh, 7).exec(dh, dh_tmp.p, -1, (R)1, s);
}

template <typename R>
bool ConvEngine<R>::contract_form() const {
  if (sigma_unfused() || sigma_ungrouped() || sigma_accum_form()) return false;
  if (op.No > 4 || !p4->reversal_ok()) return false;
  std::vector<int> ytab;
  return grouped_table(ytab);
}

template <typename R>
std::vector<typename ConvEngine<R>::SigmaGroup> ConvEngine<R>::plan_sigma(bool share, int outs, int slots) const {
  const int No = op.No, Nchi = op.Nchi;
  std::vector<SigmaGroup> P;
  std::vector<char> done((size_t)No * No, 0);
  for (int l1 = 0; l1 < No; ++l1)
    for (int m1 = 0; m1 < No; ++m1) {
      const int o = m1 + No * l1;
      if (done[o]) continue;
      std::vector<int> batch{o};
      if (share && m1 != l1) batch.push_back(l1 + No * m1);
      SigmaGroup B;
      std::map<std::pair<int, int>, int> slot;  // (m, l) -> head slot of this batch
      for (int ob : batch) {
        const int bm1 = ob % No, bl1 = ob / No;
        std::vector<std::array<int, 3>> srcl;
        for (int l = 0; l < Nchi; ++l)
          for (int m = 0; m < Nchi; ++m) {
            if (op.ol[m][0] != bm1 || op.ol[l][0] != bl1) continue;
            int e;
            auto it = slot.find({m, l});
            if (it != slot.end()) {
              e = 2 * it->second;
            } else if (share && (it = slot.find({l, m})) != slot.end()) {
              e = 2 * it->second + 1;
            } else {
              const int sl = (int)slot.size();
              slot[{m, l}] = sl;
              B.heads.push_back({m, l});
              e = 2 * sl;
            }
            srcl.push_back({m, l, e});
          }
        B.outs.push_back(ob);
        B.src.push_back(srcl);
        done[ob] = 1;
      }
      // joined to the last group while that stays within its outputs and slots
      // (outputs without a source stay apart: they are only zeroed)
      if (!P.empty() && !B.heads.empty() && !P.back().heads.empty() &&
          (int)(P.back().outs.size() + B.outs.size()) <= std::max(outs, 1) &&
          (int)(P.back().heads.size() + B.heads.size()) <= slots) {
        SigmaGroup& G = P.back();
        const int base = (int)G.heads.size();
        for (auto& sl : B.src)
          for (auto& e : sl) e[2] += 2 * base;
        G.outs.insert(G.outs.end(), B.outs.begin(), B.outs.end());
        G.src.insert(G.src.end(), B.src.begin(), B.src.end());
        G.heads.insert(G.heads.end(), B.heads.begin(), B.heads.end());
      } else {
        P.push_back(std::move(B));
      }
    }
  return P;
}

template <typename R>
void ConvEngine<R>::sigma(zd* sig, const zd* V, const double* S_h, const double* C_h, double temp, hipStream_t s,
                          bool apply_threshold) {
  // the nu -> infinity slot of V_sigma is 1.5 S - 0.5 C (fself.f90:208)
  const int Nchi = op.Nchi;
  std::vector<double> stat((size_t)Nchi * Nchi);
  for (size_t e = 0; e < stat.size(); ++e) stat[e] = 1.5 * S_h[e] - 0.5 * C_h[e];
  sigma(sig, V, stat.data(), temp, s, apply_threshold);
}

// The tables of sigma() for one static part: built on first use and when it
// or the transformed G's place changes
template <typename R>
void ConvEngine<R>::sigma_tables(const double* stat_h, hipStream_t s) {
  const int No = op.No, Nchi = op.Nchi;
  const std::vector<double> st(stat_h, stat_h + (size_t)Nchi * Nchi);
  const bool unfused = sigma_unfused();
  if (!sig_groups.empty() && st == sig_stat && sig_fg == Fg.p && sig_unfused == unfused) return;
  sig_stat = st;
  sig_fg = Fg.p;
  sig_unfused = unfused;
  // the accumulating last pass sums the pairs of one output in registers;
  // shapes it does not cover (and GMOD_SIGMA_UNFUSED=1) transform every
  // source whole and sum them in one streaming kernel
  sig_fused = p4->accum_ok(-1) && !unfused;
  // transposed outputs share their sources' head passes when the static
  // slot is symmetric (the conjugate-reversal relation of the sources, with
  // the slot-0 correction)
  bool share = sig_fused && p4->accum_last_is_t(-1) && p4->reversal_ok();
  for (int l = 0; l < Nchi && share; ++l)
    for (int m = 0; m < Nchi; ++m)
      if (stat_h[m + Nchi * l] != stat_h[l + Nchi * m]) { share = false; break; }
  // as many outputs at once as give the CUs several rounds of boxes, their
  // sources within 4 GB; a single output of the unfused form whose sources
  // exceed that is summed in parts
  sig_cap = (int)std::min<long>(std::max<long>(1, (4L << 30) / (N * (long)sizeof(cpx<R>))), 1 << 20);
  sig_groups = plan_sigma(share, p4->batch_items(No * No), sig_cap);
  std::vector<int> smap, off, heads, ta, tb, gat;
  std::vector<double> hstat;
  std::vector<long> hoffs;
  std::vector<cpx<R>*> fg;
  sig_slots = 0;
  sig_outs = 0;
  for (auto& g : sig_groups) {
    g.first_off = (int)off.size();
    g.first_src = (int)smap.size();
    g.first_head = (int)heads.size() / 2;
    g.first_out = (int)gat.size() / 4;
    const int nh = (int)g.heads.size();
    const bool parts = !sig_fused && nh > sig_cap;  // one output, a head per source
    off.push_back(0);
    int c = 0;
    for (size_t i = 0; i < g.outs.size(); ++i) {
      for (auto& e : g.src[i]) {
        if (parts && c > 0 && c % sig_cap == 0) off.push_back(c);
        const int ab = op.ol[e[0]][1] + No * op.ol[e[1]][1];
        fg.push_back(Fg.p + (long)ab * N);
        smap.push_back(e[2]);
        ta.push_back((e[2] >> 1) % (parts ? sig_cap : nh));
        tb.push_back(ab);
        ++c;
      }
      off.push_back(c);
      const int gt[4] = {g.outs[i], -1, 0, 0};
      gat.insert(gat.end(), gt, gt + 4);
    }
    g.nsrc = c;
    for (auto& h : g.heads) {
      heads.push_back(h[0] + Nchi * h[1]);
      heads.push_back(h[1] + Nchi * h[0]);
      hstat.push_back(stat_h[h[0] + Nchi * h[1]]);
      head_offsets(hoffs, h[0], h[1]);
    }
    sig_slots = std::max(sig_slots, parts ? sig_cap : nh);
    sig_outs = std::max(sig_outs, (int)g.outs.size());
  }
  sig_off.set(std::move(off), s);
  sig_map.set(std::move(smap), s);
  sig_heads.set(std::move(heads), s);
  sig_hstat.set(std::move(hstat), s);
  sig_hoffs.set(std::move(hoffs), s);
  sig_ta.set(std::move(ta), s);
  sig_tb.set(std::move(tb), s);
  sig_gat.set(std::move(gat), s);
  sig_tab.alloc(fg.size());
  sig_tab.upload(fg.data(), fg.size(), s);
  GMOD_HIP(hipStreamSynchronize(s));  // fg is released here
}

template <typename R>
void ConvEngine<R>::sigma(zd* sig, const zd* V, const double* stat_h, double temp, hipStream_t s,
                          bool apply_threshold) {
  const int No = op.No;
  const long NkNw = mesh.Nk * (long)mesh.Nw;
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  const R invN = (R)(1.0 / (double)p4->transformed_points());
  sigma_tables(stat_h, s);
  if (srcs.n < (size_t)sig_slots * N) srcs.alloc((size_t)sig_slots * N);
  if (acc.n < (size_t)sig_outs * N) acc.alloc((size_t)sig_outs * N);
  if (!mesh.complete) GMOD_HIP(hipMemsetAsync(sig, 0, NkNw * No * No * sizeof(zd), s));
  const GatherBatch<R> gat{sig, NkNw, sig_gat.ptr(),
                           GatherStore<R>{sig, temp / (double)mesh.Nkall, nullptr, nullptr, 0, md}};
  const BosonBatch<R> heads{V, NkNw, sig_heads.ptr(), sig_hstat.ptr(), md};
  for (const SigmaGroup& g : sig_groups) {
    const int nh = (int)g.heads.size(), no = (int)g.outs.size();
    if (g.nsrc == 0) {
      for (int o : g.outs) GMOD_HIP(hipMemsetAsync(sig + NkNw * o, 0, NkNw * sizeof(zd), s));
      continue;
    }
    if (sig_fused) {
      p4->exec_head(heads.from(g.first_head), srcs.p, nh, tmp.p, -1, s);
      if (dhD.n < (size_t)nh * S) dhD.alloc((size_t)nh * S);
      slot0_corr(dhD.p, V, sig_hoffs.d.p + 2 * (long)g.first_head, nh, s);
      p4->exec_accum_last(srcs.p, N, g.nsrc, MulAccAccum<R>{sig_tab.p + g.first_src, acc.p, S, N}, -1, (R)1, s,
                          sig_map.d.p + g.first_src, dhD.p, sig_off.d.p + g.first_off, no);
    } else {
      for (int h0 = 0, part = 0; h0 < nh; h0 += sig_cap, ++part) {
        p4->exec_batch(heads.from(g.first_head + h0), GridStore<R>{srcs.p, S, N}, srcs.p, std::min(sig_cap, nh - h0),
                       tmp.p, -1, (R)1, s);
        contract<R>(acc.p, srcs.p, Fg.p, sig_off.d.p + g.first_off + part, sig_ta.d.p + g.first_src,
                    sig_tb.d.p + g.first_src, no, N, part > 0, s);
      }
    }
    p4->exec_batch(GridLoad<R>{acc.p, S, N}, gat.from(g.first_out), acc.p, no, tmp.p, +1, invN, s);
  }
  if (apply_threshold) threshold(sig, NkNw * No * No, 1e-9, s);
}

template <typename R>
void ConvEngine<R>::prepare_gap(const zd* Vd, const double* S_h, const double* C_h, bool singlet, hipStream_t s) {
  const int Nchi = op.Nchi;
  const double sgn = singlet ? 1.0 : -1.0;
  gap_pairs.clear();
  for (int l = 0; l < Nchi; ++l)
    for (int m = 0; m < Nchi; ++m)
      if (op.ol[l][0] >= op.ol[m][1]) gap_pairs.push_back({l, m});
  {
    std::vector<int> heads, off{0}, ta, tb, gat;
    std::vector<double> stat;
    for (auto& p : gap_pairs) {
      const int l = p[0], m = p[1];
      heads.push_back(m + Nchi * l);
      heads.push_back(l + Nchi * m);
      stat.push_back(0.5 * (S_h[m + Nchi * l] + sgn * C_h[m + Nchi * l]));
    }
    for (int m2 = 0; m2 < op.No; ++m2)
      for (int l1 = 0; l1 < op.No; ++l1) {
        for (size_t q = 0; q < gap_pairs.size(); ++q) {
          const int l = gap_pairs[q][0], m = gap_pairs[q][1];
          if (op.ol[l][0] != l1 || op.ol[m][1] != m2) continue;
          ta.push_back((int)q);
          tb.push_back(op.ol[l][1] + op.No * op.ol[m][0]);
        }
        if ((int)ta.size() == off.back()) continue;
        off.push_back((int)ta.size());
        const int g[4] = {l1 + op.No * m2, -1, 0, 0};
        gat.insert(gat.end(), g, g + 4);
      }
    gap_heads.set(std::move(heads), s);
    gap_stat.set(std::move(stat), s);
    gap_off.set(std::move(off), s);
    gap_ta.set(std::move(ta), s);
    gap_tb.set(std::move(tb), s);
    gap_gat.set(std::move(gat), s);
  }
  Vd_dev = Vd;
  size_t free_b = 0, total_b = 0;
  GMOD_HIP(hipMemGetInfo(&free_b, &total_b));
  const double need = (double)gap_pairs.size() * N * sizeof(cpx<R>);
  vft_cached = need < 0.5 * (double)free_b;
  if (!vft_cached) return;
  if (Vft.n != gap_pairs.size() * (size_t)N) Vft.alloc(gap_pairs.size() * (size_t)N);
  const int n = (int)gap_pairs.size(), step = p4->batch_items(n);
  for (int i0 = 0; i0 < n; i0 += step) {
    cpx<R>* g = Vft.p + (long)i0 * N;
    p4->exec_batch(gap_boson(Vd).from(i0), GridStore<R>{g, (unsigned)mesh.Nkall, N}, g, std::min(step, n - i0), tmp.p,
                   -1, (R)1, s);
  }
}

template <typename R>
BosonBatch<R> ConvEngine<R>::gap_boson(const zd* Vd) const {
  return BosonBatch<R>{Vd, mesh.Nk * (long)mesh.Nw, gap_heads.ptr(), gap_stat.ptr(), mesh_dev(mesh)};
}

template <typename R>
void ConvEngine<R>::gap(zd* nd, const zd* F, const double* prt, bool singlet, double weight, hipStream_t s) {
  const int No = op.No;
  const long NkNw = mesh.Nk * (long)mesh.Nw;
  const double sgn = singlet ? 1.0 : -1.0, dprt = sgn;
  if (Ff.n != (size_t)(No * No) * N) Ff.alloc((size_t)No * No * N);
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  const R invN = (R)(1.0 / (double)p4->transformed_points());
  if (gap_prt.h != std::vector<double>(prt, prt + No)) gap_prt.set(std::vector<double>(prt, prt + No), s);
  p4->exec_batch(AnomBatch<R>{F, NkNw, No, gap_prt.ptr(), sgn, dprt, md}, GridStore<R>{Ff.p, S, N}, Ff.p, No * No, tmp.p,
                 -1, (R)1, s);
  GMOD_HIP(hipMemsetAsync(nd, 0, NkNw * No * No * sizeof(zd), s));
  // the outputs (l1, m2) that have pairs, their products summed in pair order
  const int nout = (int)gap_gat.h.size() / 4, step = p4->batch_items(nout);
  if (acc.n < (size_t)step * N) acc.alloc((size_t)step * N);
  const GatherBatch<R> gat{nd, NkNw, gap_gat.ptr(), GatherStore<R>{nd, weight, nullptr, nullptr, 0, md}};
  for (int o0 = 0; o0 < nout; o0 += step) {
    const int no = std::min(step, nout - o0);
    if (vft_cached) {
      contract<R>(acc.p, Vft.p, Ff.p, gap_off.d.p + o0, gap_ta.d.p, gap_tb.d.p, no, N, false, s);
    } else {
      for (int o = o0; o < o0 + no; ++o)
        for (int c = gap_off.h[o]; c < gap_off.h[o + 1]; ++c)
          p4->exec_fused(gap_boson(Vd_dev).from(gap_ta.h[c]),
                         MulAccStore<R>{acc.p + (long)(o - o0) * N, Ff.p + (long)gap_tb.h[c] * N,
                                        c == gap_off.h[o] ? 1 : 0, S},
                         work.p, tmp.p, -1, (R)1, s);
    }
    p4->exec_batch(GridLoad<R>{acc.p, S, N}, gat.from(o0), acc.p, no, tmp.p, +1, invN, s);
  }
  hermitize_lower(nd, mesh.Nk, mesh.Nw, No, s);
}

template <typename R>
void ConvEngine<R>::prepare_gap_soc(const zd* Vd, const double* Vmat_h, const int64_t* invschi, long gap_sym,
                                    hipStream_t s) {
  if (!op.soc) throw Error("prepare_gap_soc: the orbital pairs carry no spin");
  if (!mesh.nfull_ok) throw Error("lin_eliash_soc: invk(3,:) must give the -k point of every k");
  const int Nchi = op.Nchi;
  const long NC = mesh.Nk * (long)mesh.Nw;
  const MeshDev md = mesh_dev(mesh);
  // the pairs of feliashwithsoc.f90:538-540: every spin for a triplet gap,
  // opposite spins of (l1, m2) for a singlet; of those the up-l1 ones (or,
  // for the parity-mixed gap_sym = -10, every opposite-spin one), and of the
  // opposite-spin ones the upper triangle l1 >= -m2
  gap_pairs.clear();
  soc_vload.clear();
  for (int l = 0; l < Nchi; ++l)
    for (int m = 0; m < Nchi; ++m) {
      const int l1 = op.ol[l][0], m2 = op.ol[m][1];
      const double ss = op.spin[l1] * op.spin[m2];
      if (!(gap_sym < 0 || (gap_sym > 0 && ss < 0))) continue;
      if (!((gap_sym == -10 && ss < 0) || op.spin[l1] > 0)) continue;
      if (!(op.spin[m2] > 0 || l1 >= op.inv[m2])) continue;
      const long li = invschi[l] - 1, mi = invschi[m] - 1;
      if (li < 0 || li >= Nchi || mi < 0 || mi >= Nchi) throw Error("lin_eliash_soc: invschi entry outside [1,Nchi]");
      gap_pairs.push_back({l, m});
      soc_vload.push_back(SocBosonLoad<R>{Vd, NC * (m + (long)Nchi * l), NC * (l + (long)Nchi * m),
                                          NC * (li + (long)Nchi * mi), NC * (mi + (long)Nchi * li),
                                          op.psign[m + Nchi * l], zd(-Vmat_h[m + Nchi * l], 0), md});
    }
  size_t free_b = 0, total_b = 0;
  GMOD_HIP(hipMemGetInfo(&free_b, &total_b));
  const double need = (double)gap_pairs.size() * N * sizeof(cpx<R>);
  vft_cached = need < 0.5 * (double)free_b;
  if (!vft_cached) return;
  Vft.alloc(gap_pairs.size() * (size_t)N);
  for (size_t q = 0; q < gap_pairs.size(); ++q) {
    cpx<R>* g = Vft.p + q * N;
    p4->exec_fused(soc_vload[q], GridStore<R>{g, (unsigned)mesh.Nkall}, g, tmp.p, -1, (R)1, s);
  }
}

template <typename R>
void ConvEngine<R>::gap_soc(zd* nd, const zd* F, hipStream_t s) {
  const int No = op.No;
  const long NW = mesh.Nkall * (long)mesh.Nw;
  if (Ff.n != (size_t)(No * No) * N) Ff.alloc((size_t)No * No * N);
  if (acc.n < (size_t)N) acc.alloc(N);
  const MeshDev md = mesh_dev(mesh);
  const R invN = (R)(1.0 / (double)p4->transformed_points());
  std::vector<char> need((size_t)No * No, 0);
  for (auto& lm : gap_pairs) need[op.ol[lm[0]][1] + No * op.ol[lm[1]][0]] = 1;
  for (int b = 0; b < No; ++b)
    for (int a = 0; a < No; ++a) {
      if (!need[a + No * b]) continue;
      cpx<R>* g = grid(Ff, a, b);
      p4->exec_fused(FullAnomLoad<R>{F, NW * (a + (long)No * b), NW * (b + (long)No * a), md},
                     GridStore<R>{g, (unsigned)mesh.Nkall}, g, tmp.p, -1, (R)1, s);
    }
  GMOD_HIP(hipMemsetAsync(nd, 0, NW * No * No * sizeof(zd), s));
  for (int m2 = 0; m2 < No; ++m2)
    for (int l1 = 0; l1 < No; ++l1) {
      bool first = true;
      for (size_t q = 0; q < gap_pairs.size(); ++q) {
        const int l = gap_pairs[q][0], m = gap_pairs[q][1];
        if (op.ol[l][0] != l1 || op.ol[m][1] != m2) continue;
        const cpx<R>* fg = grid(Ff, op.ol[l][1], op.ol[m][0]);
        if (vft_cached)
          mul_acc<R>(acc.p, Vft.p + q * N, fg, first, N, s);
        else
          p4->exec_fused(soc_vload[q], MulAccStore<R>{acc.p, fg, first ? 1 : 0, (unsigned)mesh.Nkall}, work.p,
                         tmp.p, -1, (R)1, s);
        first = false;
      }
      if (first) continue;
      p4->exec_fused(GridLoad<R>{acc.p, (unsigned)mesh.Nkall}, FullGatherStore<R>{nd + NW * (l1 + (long)No * m2), 0, md},
                     acc.p, tmp.p, +1, invN, s);
    }
}

// ====================================================================== increments
// Rolling increments for the mixed-precision FLEX loop.  Between iterations
// n-1 and n the bubble and the self-energy change by
//   dB = B(Gr + dG) - B(Gr)  = dG13 (Gr42 + dG42) + Gr13 dG42      (per product)
//   dS = S(Vr + dV, Gr + dG) - S(Vr, Gr) = dV (Gr + dG) + Vr dG
// with Gr, Vr the previous iterate.  dG and dV are formed in FP64 in k-space
// and only the increments are transformed at the grid precision, so the
// rounding error of an update is proportional to the update itself and
// vanishes as the loop converges; the transforms of the previous iterate
// (Fr, F0r, TAr, TBr, FVr) advance by the transformed increments.
template <typename R>
void ConvEngine<R>::set_reference(const zd* Gref, const zd* G0ref, bool tail, const double* eig_d, const zd* uni_d,
                                  double mu_ref, double temp, hipStream_t s) {
  const int No = op.No;
  const size_t nb = (size_t)No * No * N;
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  auto ensure = [&](DBuf<cpx<R>>& b) { if (b.n != nb) b.alloc(nb); };
  ensure(Fr); ensure(Fd);
  p4->exec_batch(GreenBatch<R>{Gref, No, md}, GridStore<R>{Fr.p, S, N}, Fr.p, No * No, tmp.p, -1, (R)1, s);
  if (!tail) return;
  ensure(F0r); ensure(F0d); ensure(TAr); ensure(TBr); ensure(TAd); ensure(TBd);
  p4->exec_batch(GreenBatch<R>{G0ref, No, md}, GridStore<R>{F0r.p, S, N}, F0r.p, No * No, tmp.p, -1, (R)1, s);
  tau_grids(TAr.p, TBr.p, eig_d, uni_d, mu_ref, mu_ref, false, temp, s);
}

template <typename R>
void ConvEngine<R>::set_vertex_reference(const zd* Vref, const double* S_h, const double* C_h, hipStream_t s) {
  const int Nchi = op.Nchi;
  const long NC = mesh.Nk * (long)mesh.Nw;
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  // the static slot 3/2 S - 1/2 C must be symmetric for the transposed pair
  // to be the conjugate reversal
  bool share = contract_form();
  for (int l = 0; l < Nchi && share; ++l)
    for (int m = 0; m < Nchi; ++m)
      if (S_h[m + Nchi * l] != S_h[l + Nchi * m] || C_h[m + Nchi * l] != C_h[l + Nchi * m]) {
        share = false;
        break;
      }
  std::vector<std::array<int, 2>> heads;
  if (share) {
    heads = share_heads(fv_entry);
  } else {
    fv_entry.assign((size_t)Nchi * Nchi, 0);
    for (int l = 0; l < Nchi; ++l)
      for (int m = 0; m < Nchi; ++m) {
        fv_entry[m + Nchi * l] = 2 * (m + Nchi * l);
        heads.push_back({m, l});
      }
  }
  fv_shared = share;
  const size_t nb = heads.size() * (size_t)N;
  if (FVr.n != nb) FVr.alloc(nb);
  if (share) {
    std::vector<long> hoffs;
    for (auto& h : heads) head_offsets(hoffs, h[0], h[1]);
    if (dhF_offs.n != hoffs.size()) dhF_offs.alloc(hoffs.size());
    dhF_offs.upload(hoffs.data(), hoffs.size(), s);
    if (dhF.n != heads.size() * (size_t)mesh.Nkall) dhF.alloc(heads.size() * (size_t)mesh.Nkall);
    slot0_corr(dhF.p, Vref, dhF_offs.p, (int)heads.size(), s);
    GMOD_HIP(hipStreamSynchronize(s));  // hoffs is released here
  }
  std::vector<int> sl;
  std::vector<double> st;
  for (auto& h : heads) {
    const int m = h[0], l = h[1];
    sl.push_back(m + Nchi * l);
    sl.push_back(l + Nchi * m);
    st.push_back(1.5 * S_h[m + Nchi * l] - 0.5 * C_h[m + Nchi * l]);
  }
  fv_heads.set(std::move(sl), s);
  fv_stat.set(std::move(st), s);
  const BosonBatch<R> bb{Vref, NC, fv_heads.ptr(), fv_stat.ptr(), md};
  const int n = (int)heads.size(), step = p4->batch_items(n);
  for (int i0 = 0; i0 < n; i0 += step) {
    cpx<R>* g = FVr.p + (long)i0 * N;
    p4->exec_batch(bb.from(i0), GridStore<R>{g, S, N}, g, std::min(step, n - i0), tmp.p, -1, (R)1, s);
  }
}

template <typename R>
void ConvEngine<R>::chi0_increment(zd* chi, const zd* chi_base, const zd* G, const zd* Gref, const zd* G0,
                                   const zd* G0ref, double temp, bool tail, const double* eig_d, const zd* uni_d,
                                   double mu, double mu_ref, const zd* dJ, const zd* sawc_d,
                                   hipStream_t s) {
  const int No = op.No, Nchi = op.Nchi;
  const long NkNw = mesh.Nk * (long)mesh.Nw;
  const double w = temp / (double)mesh.Nkall;
  const double wref = 1.0 / (temp * (double)mesh.Nkall);
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  const R invN = (R)(1.0 / (double)p4->transformed_points());
  // the Green-function differences in FP64 and rounded to the grid's FP32
  // once in k space (the values the difference load forms per grid point),
  // then transformed from a quarter of the bytes
  const long nG = NkNw * No * No;
  auto diff_pass = [&](const zd* X, const zd* Xref, DBuf<cpx<R>>& F) {
    if constexpr (sizeof(R) == 4) {
      if (dgbuf.n != (size_t)nG) dgbuf.alloc(nG);
      diff_to_f32(dgbuf.p, X, Xref, nG, s);
      p4->exec_batch(GreenBatch<R, float>{dgbuf.p, No, md}, GridStore<R>{F.p, S, N}, F.p, No * No, tmp.p, -1, (R)1, s);
    } else {
      throw Error("chi0_increment: FP32 transforms only");
    }
  };
  diff_pass(G, Gref, Fd);
  if (tail) {
    diff_pass(G0, G0ref, F0d);
    tau_grids(TAd.p, TBd.p, eig_d, uni_d, mu, mu_ref, true, temp, s);
  }
  // (mirrored copies as in chi0 measured no faster here: the 2 No^2 copies
  // per iteration cost what the in-place reads save, and the spatial-first
  // inverse reads the (-r,-t) operands as whole reversed planes)
  const bool fuse = mesh.complete;
  auto gather = [&](const PairTab& t, double wt, bool jumps, const zd* base, int acc_) {
    GatherStore<R> g = gather_sf(chi, wt, jumps ? dJ : nullptr, jumps ? sawc_d : nullptr, acc_, s);
    g.base = base;
    return GatherBatch<R>{chi, NkNw, t.gat.ptr(), g};
  };
  const PairTab& t = fuse ? pairs_other : other_plain;
  if (tail) {
    const R mw = (R)(-w), pw = (R)w, mr = (R)(-wref);
    product_batches(IncProductBatch<R, 3>{{Fr.p, F0r.p, TAr.p}, {Fd.p, F0d.p, TAd.p}, {Fr.p, F0r.p, TBr.p},
                                          {Fd.p, F0d.p, TBd.p}, {mw, pw, mr}, {1, 1, 0}, N, t.prod.ptr(), md},
                    gather(t, 1.0, true, chi_base, 0), t.n, s);
    // a self-partner pair: the increment of conj(conv[G] + ref) - conv[G0]
    product_batches(IncProductBatch<R, 2>{{Fr.p, TAr.p}, {Fd.p, TAd.p}, {Fr.p, TBr.p}, {Fd.p, TBd.p}, {mw, mr}, {1, 0},
                                          N, pairs_self.prod.ptr(), md},
                    gather(pairs_self, 1.0, true, chi_base, 0), pairs_self.n, s);
    product_batches(IncProductBatch<R, 1>{{F0r.p}, {F0d.p}, {F0r.p}, {F0d.p}, {pw}, {1}, N, self_plain.prod.ptr(), md},
                    gather(self_plain, 1.0, false, nullptr, 1), self_plain.n, s);
  } else {
    // (the reference conjugates a self-partner pair in place after the
    // accumulation, fchi.f90:610: the stored value is conj(conv[G]), so the
    // increment is conjugated before it is added)
    auto inc = [&](const PairTab& q) {
      return IncProductBatch<R, 1>{{Fr.p}, {Fd.p}, {Fr.p}, {Fd.p}, {(R)-1}, {1}, N, q.prod.ptr(), md};
    };
    product_batches(inc(t), gather(t, w, false, chi_base, 0), t.n, s);
    product_batches(inc(pairs_self), gather(pairs_self, w, false, chi_base, 0), pairs_self.n, s);
  }
  if (!fuse) partner_copies(chi, pairs_other.gat.d.p, pairs_other.n, NkNw, s);
}

template <typename R>
void ConvEngine<R>::sigma_increment(zd* sig, const zd* sig_base, const zd* V, const zd* Vref, double temp,
                                    hipStream_t s, bool dv_ready) {
  const int No = op.No, Nchi = op.Nchi;
  const long NkNw = mesh.Nk * (long)mesh.Nw;
  if (acc.n < (size_t)N) acc.alloc(N);
  const MeshDev md = mesh_dev(mesh);
  const unsigned S = (unsigned)mesh.Nkall;
  const R invN = (R)(1.0 / (double)p4->transformed_points());
  const long NC = NkNw;
  // the vertex difference once in k space at grid precision: each element is
  // then read (from a quarter of the bytes) by the four grid points that
  // unfold it, instead of two FP64 reads per grid point
  const long nC = NkNw * Nchi * Nchi;
  if (!dv_ready || dvbuf.n != (size_t)nC) {
    if (dvbuf.n != (size_t)nC) dvbuf.alloc(nC);
    diff_to_f32(dvbuf.p, V, Vref, nC, s);
  }
  // the inverse transform of output (m1, l1) from grid g, gathered onto sig_base + sig
  auto gather_out = [&](int m1, int l1) {
    GatherBatch<R> gat{sig, NkNw, orb_gat.ptr(),
                       GatherStore<R>{sig, temp / (double)mesh.Nkall, nullptr, nullptr, 0, md}};
    gat.proto.base = sig_base;
    p4->exec_batch(GridLoad<R>{acc.p, S, N}, gat.from(m1 + No * l1), acc.p, 1, tmp.p, +1, invN, s);
  };
  // every pair's slices, for the forms that transform pair by pair
  if (all_heads.h.empty()) {
    std::vector<int> sl;
    for (int l = 0; l < Nchi; ++l)
      for (int m = 0; m < Nchi; ++m) {
        sl.push_back(m + Nchi * l);
        sl.push_back(l + Nchi * m);
      }
    all_heads.set(std::move(sl), s);
  }
  auto pair_load = [&](int m, int l) {
    return BosonBatch<R, float>{dvbuf.p, NC, all_heads.ptr(), DualPtr<double>{}, md}.from(m + (long)Nchi * l);
  };
  std::vector<int> ytab;
  if (contract_form()) {
    // contraction form: the full transform of every vertex difference once
    // per transposed pair, then all outputs in one streaming kernel
    grouped_table(ytab);
    std::vector<int> dent;
    const std::vector<std::array<int, 2>> heads = share_heads(dent);
    const size_t nb = heads.size() * (size_t)N;
    if (DVt.n != nb) DVt.alloc(nb);
    if (dv_heads.h.empty()) {
      std::vector<int> sl;
      for (auto& h : heads) {
        sl.push_back(h[0] + Nchi * h[1]);
        sl.push_back(h[1] + Nchi * h[0]);
      }
      dv_heads.set(std::move(sl), s);
    }
    const BosonBatch<R, float> bb{dvbuf.p, NC, dv_heads.ptr(), DualPtr<double>{}, md};
    const int n = (int)heads.size(), step = p4->batch_items(n);
    for (int i0 = 0; i0 < n; i0 += step) {
      cpx<R>* g = DVt.p + (long)i0 * N;
      p4->exec_batch(bb.from(i0), GridStore<R>{g, S, N}, g, std::min(step, n - i0), tmp.p, -1, (R)1, s);
    }
    {
      std::vector<long> hoffs;
      for (auto& h : heads) head_offsets(hoffs, h[0], h[1]);
      if (dh_offs.n < hoffs.size()) dh_offs.alloc(hoffs.size());
      dh_offs.upload(hoffs.data(), hoffs.size(), s);
      if (dhD.n < heads.size() * (size_t)mesh.Nkall) dhD.alloc(heads.size() * (size_t)mesh.Nkall);
      slot0_corr(dhD.p, (const cpx<float>*)dvbuf.p, dh_offs.p, (int)heads.size(), s);
      GMOD_HIP(hipStreamSynchronize(s));  // hoffs is released here
    }
    const int NAB = No * No;
    if (fv_entry.size() != (size_t)Nchi * Nchi) throw Error("sigma_increment: no reference vertex transforms");
    std::vector<int> ct(2 * ytab.size());
    for (size_t i = 0; i < ytab.size(); ++i) {
      ct[2 * i] = fv_entry[ytab[i]];
      ct[2 * i + 1] = dent[ytab[i]];
    }
    if (ctab_d.n != ct.size()) ctab_d.alloc(ct.size());
    ctab_d.upload(ct.data(), ct.size(), s);
    if (ysum.n < (size_t)NAB * N) ysum.alloc((size_t)NAB * N);
    {
      // per point: two vertex grids and Fd per (output, pair), Fr, one write per output
      const double per = 2.0 * NAB * NAB + 2.0 * NAB + NAB;
      ProfScope ps(sizeof(R) == 4 ? PROF_FFT32 : PROF_FFT, per * (double)N * sizeof(cpx<R>), s);
      sigma_inc_contract<R>(ysum.p, Fr.p, Fd.p, FVr.p, DVt.p, dhF.p, dhD.p, ctab_d.p, NAB, No, S, (unsigned)(N / S),
                            mesh.rev.p, s);
    }
    GMOD_HIP(hipStreamSynchronize(s));  // ct is released at return
    GatherBatch<R> gat{sig, NkNw, orb_gat.ptr(),
                       GatherStore<R>{sig, temp / (double)mesh.Nkall, nullptr, nullptr, 0, md}};
    gat.proto.base = sig_base;
    p4->exec_batch(GridLoad<R>{ysum.p, S, N}, gat, ysum.p, NAB, tmp.p, +1, invN, s);
    return;
  }
  if (fv_shared) throw Error("sigma_increment: the reference vertex transforms are stored in the contraction form");
  const bool fused = p4->accum_ok(-1) && !sigma_unfused();
  // grouped form (every output has one source per orbital pair (a, b), No <= 4):
  // the reference-vertex term Y_o = sum FVr Fd and Gn = Fr + Fd in one
  // streaming kernel, then the accumulating pass with one operand per source
  bool grouped = fused && No <= 4 && !sigma_ungrouped() && grouped_table(ytab);
  // ysum: Y of the No^2 outputs, then Gn of the No^2 orbital pairs
  if (grouped && ysum.n != (size_t)2 * No * No * N) ysum.alloc((size_t)2 * No * No * N);
  if (!fused) {
    for (int l1 = 0; l1 < No; ++l1)
      for (int m1 = 0; m1 < No; ++m1) {
        bool first = true;
        for (int l = 0; l < Nchi; ++l)
          for (int m = 0; m < Nchi; ++m) {
            if (op.ol[m][0] != m1 || op.ol[l][0] != l1) continue;
            const int a = op.ol[m][1], b = op.ol[l][1];
            SigmaIncStore<R> st{acc.p, grid(Fr, a, b), grid(Fd, a, b), FVr.p + (size_t)(m + Nchi * l) * N,
                                first ? 1 : 0, S};
            p4->exec_fused(pair_load(m, l), st, work.p, tmp.p, -1, (R)1, s);
            first = false;
          }
        if (!first) gather_out(m1, l1);
      }
    return;
  }
  // transposed outputs share the head passes of their sources (the vertex
  // differences' static slot is zero, so the conjugate-reversal relation
  // holds, with the slot-0 correction)
  const std::vector<SigmaGroup> P = plan_sigma(p4->accum_last_is_t(-1) && p4->reversal_ok(), 1, 1 << 20);
  accum_tab_h.clear();
  std::vector<int> smap;
  std::vector<long> hoffs;
  size_t nmax = 0;
  for (auto& g : P) {
    for (auto& sl : g.src)
      for (auto& e : sl) {
        const int m = e[0], l = e[1], a = op.ol[m][1], b = op.ol[l][1];
        if (grouped) {
          accum_tab_h.push_back(ysum.p + (size_t)No * No * N + (size_t)(a + No * b) * N);  // Gn_ab
        } else {
          accum_tab_h.push_back(grid(Fr, a, b));
          accum_tab_h.push_back(grid(Fd, a, b));
          accum_tab_h.push_back(FVr.p + (size_t)(m + Nchi * l) * N);
        }
        smap.push_back(e[2]);
      }
    for (auto& h : g.heads) head_offsets(hoffs, h[0], h[1]);
    nmax = std::max(nmax, g.heads.size());
  }
  if (srcs.n < nmax * N) srcs.alloc(nmax * N);
  accum_tab.alloc(accum_tab_h.size());
  accum_tab.upload(accum_tab_h.data(), accum_tab_h.size(), s);
  srcmap_d.alloc(smap.size());
  srcmap_d.upload(smap.data(), smap.size(), s);
  if (dh_offs.n < hoffs.size()) dh_offs.alloc(hoffs.size());
  if (!hoffs.empty()) dh_offs.upload(hoffs.data(), hoffs.size(), s);
  if (dhD.n < nmax * mesh.Nkall) dhD.alloc(nmax * mesh.Nkall);
  if (grouped) {
    if (ytab_d.n != ytab.size()) ytab_d.alloc(ytab.size());
    ytab_d.upload(ytab.data(), ytab.size(), s);
  }
  GMOD_HIP(hipStreamSynchronize(s));
  if (grouped) {
    const double NAB = (double)No * No;
    ProfScope ps(sizeof(R) == 4 ? PROF_FFT32 : PROF_FFT, (NAB * NAB + 4.0 * NAB) * (double)N * sizeof(cpx<R>), s);
    sigma_ref_contract<R>(ysum.p, ysum.p + (size_t)No * No * N, Fr.p, Fd.p, FVr.p, ytab_d.p, No * No, No, N, s);
  }
  long off = 0, hoff = 0;
  for (auto& g : P) {
    for (size_t h = 0; h < g.heads.size(); ++h)
      p4->exec_head(pair_load(g.heads[h][0], g.heads[h][1]), srcs.p + (long)h * N, 1, tmp.p, -1, s);
    slot0_corr(dhD.p, (const cpx<float>*)dvbuf.p, dh_offs.p + 2 * hoff, (int)g.heads.size(), s);
    hoff += (long)g.heads.size();
    for (size_t i = 0; i < g.outs.size(); ++i) {
      const int nsrc = (int)g.src[i].size(), o = g.outs[i];
      if (nsrc == 0) continue;
      if (grouped) {
        p4->exec_accum_last(srcs.p, N, nsrc, SigmaIncAccumG<R>{accum_tab.p + off, ysum.p + (size_t)o * N, acc.p, S}, -1,
                            (R)1, s, srcmap_d.p + off, dhD.p);
      } else {
        p4->exec_accum_last(srcs.p, N, nsrc, SigmaIncAccum<R>{accum_tab.p + 3 * off, acc.p, S}, -1, (R)1, s,
                            srcmap_d.p + off, dhD.p);
      }
      off += nsrc;
      gather_out(o % No, o / No);
    }
  }
}

}  // namespace gmod
