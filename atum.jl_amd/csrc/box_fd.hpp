// Entropy-conservative flux differencing in the reference's :per_dir order (src/dgsem.jl:470-561) on box
// elements: fd_body with the compact geometry.
//
// The sums keep the reference's order, every product and sum rounded; with a diagonal metric only row
// r of the two-point flux enters direction r, a third of the products.  Quotients and square roots are
// fast_div and fast_sqrt, which round as IEEE's do, by reciprocals that the pair's or node's quotients
// share; the logarithm of the logarithmic means is lm_logavg's (a seventh of the instructions of
// the library's, and as close).  Every value equals the general kernels' but for the last bit of
// that logarithm.
#pragma once
#include "box.hpp"
#include "log_mean.hpp"

namespace atm {

// One side of a face: velocity, own pressure and 1/rho, rounded as the laws' flux() and pressure()
template <class L>
struct RefSide {
  static constexpr int D = L::D;
  static constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  double ir, u[D], e, p;  // e: rho e - rho |u|^2/2
  ATM_DEV RefSide(const LawConst& c, const double* q, const double* a) {
    ir = fast_rcp(q[0]);
#pragma unroll
    for (int d = 0; d < D; ++d) u[d] = fast_div(q[1 + d], q[0], ir);
    e = q[D + 1] - fast_div(dotv<D>(q + 1, q + 1), 2 * q[0], 0.5 * ir);
    p = pressure(c, q, GRAV ? a[0] : 0.0);
  }
  ATM_DEV double pressure(const LawConst& c, const double* q, double phi) const {
    return GRAV ? (c.gamma - 1) * (e - q[0] * phi) : (c.gamma - 1) * e;
  }
  ATM_DEV double soundspeed(const LawConst& c, const double* q, double pressure) const {
    return fast_sqrt(fast_div(c.gamma * pressure, q[0], ir));
  }
  // row R of the physical flux
  template <int R>
  ATM_DEV void flux(const LawConst& c, const double* q, const double* a, double* F) const {
    double dp = p;
    if (GRAV && c.pde_level_balance) dp -= a[D + 2];
    F[0] = q[1 + R];
#pragma unroll
    for (int e = 0; e < D; ++e) F[1 + e] = e == R ? q[1 + R] * u[e] + dp : q[1 + R] * u[e];
    F[D + 1] = u[R] * (q[D + 1] + p);
  }
};

// surfaceflux<L, SF> of the Euler laws with the normal sg * e_R in the reference's order (laws.hpp), the
// products with the normal's zeros left out
template <class L, int SF, int R>
ATM_DEV void axis_ref_flux(const LawConst& c, double sg, const double* qm, const double* am, const double* qp,
                           const double* ap, double* nf) {
  constexpr int D = L::D, Ns = L::Ns;
  constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  const RefSide<L> M(c, qm, am), P(c, qp, ap);
  double Fm[Ns], Fp[Ns];
  M.template flux<R>(c, qm, am, Fm);
  P.template flux<R>(c, qp, ap, Fp);
  if constexpr (SF == ATM_FLUX_RUSANOV) {
    const double ws = fmax(fabs(M.u[R]) + M.soundspeed(c, qm, M.p), fabs(P.u[R]) + P.soundspeed(c, qp, P.p));
#pragma unroll
    for (int s = 0; s < Ns; ++s) nf[s] = sg * ((Fm[s] + Fp[s]) / 2) - ws * (qp[s] - qm[s]) / 2;
  } else {
    static_assert(SF == ATM_FLUX_ROE, "Rusanov or Roe");
    const double phi = GRAV ? am[0] : 0.0;
    const double pm = M.p, pp = GRAV ? P.pressure(c, qp, phi) : P.p;
    const double hm = fast_div(qm[D + 1], qm[0], M.ir) + fast_div(pm, qm[0], M.ir);
    const double hp = fast_div(qp[D + 1], qp[0], P.ir) + fast_div(pp, qp[0], P.ir);
    const double cm = M.soundspeed(c, qm, pm), cp = P.soundspeed(c, qp, pp);
    const double rho = fast_sqrt(qm[0] * qp[0]);
    const double sm = fast_sqrt(qm[0]), sp = fast_sqrt(qp[0]), den = sm + sp, iden = fast_rcp(den);
    auto mean = [&](double a, double b) { return fast_div(sm * a + sp * b, den, iden); };
    double u[D], du[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      u[d] = mean(M.u[d], P.u[d]);
      du[d] = P.u[d] - M.u[d];
    }
    const double h = mean(hm, hp), cs = mean(cm, cp);
    const double un = sg * u[R], dun = sg * du[R];
    const double drho = qp[0] - qm[0], dp = pp - pm;
    const double cm2 = fast_rcp(cs * cs);
    const double w1 = fabs(un - cs) * (dp - rho * cs * dun) * cm2 / 2;
    const double w2 = fabs(un + cs) * (dp + rho * cs * dun) * cm2 / 2;
    const double w3 = fabs(un) * (drho - dp * cm2);
    const double w4 = fabs(un) * rho;
    double fp[Ns];
    fp[0] = (w1 + w2 + w3) / 2;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (d == R) fp[1 + d] = (w1 * (u[d] - cs * sg) + w2 * (u[d] + cs * sg) + w3 * u[d]) / 2;
      else fp[1 + d] = (w1 * u[d] + w2 * u[d] + w3 * u[d] + w4 * du[d]) / 2;
    }
    double e3;
    if (GRAV) {
      e3 = w3 * (dotv<D>(u, u) / 2 + phi);
    } else {
      double w3u[D];
#pragma unroll
      for (int d = 0; d < D; ++d) w3u[d] = w3 * u[d];
      e3 = dotv<D>(w3u, u) / 2;
    }
    fp[D + 1] = (w1 * (h - cs * un) + w2 * (h + cs * un) + e3 + w4 * (dotv<D>(u, du) - un * dun)) / 2;
#pragma unroll
    for (int s = 0; s < Ns; ++s) nf[s] = sg * (Fm[s] + Fp[s]) / 2 - fp[s];
  }
}

// Per-node primitives [rho, u (D), b, u.u, phi (gravity)] and, behind them in LDS, MJ
template <class L>
struct BoxPairEC {
  static constexpr int D = L::D, Ns = L::Ns;
  static constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  static constexpr int NP = GRAV ? D + 4 : D + 3;
  ATM_DEV static void prim(const LawConst& c, const double* q, const double* a, double* P) {
    const RefSide<L> S(c, q, a);
    P[0] = q[0];
#pragma unroll
    for (int d = 0; d < D; ++d) P[1 + d] = S.u[d];
    const double p2 = 2 * S.p;
    P[D + 1] = fast_div(q[0], p2, fast_rcp(p2));
    P[D + 2] = dotv<D>(S.u, S.u);
    if (GRAV) P[D + 3] = a[0];
  }
  // row R of EulerPair<D, GRAV, EC>::pair (pairflux.hpp); gm1x2: 2 (gamma - 1), ib2: 1 / 2b of node 1
  template <int R>
  ATM_DEV static void pair(double gm1x2, const double* P1, double ib2, const double* P2, double* F) {
    const double r1 = P1[0], r2 = P2[0], b1 = P1[D + 1], b2 = P2[D + 1];
    const double sr = r1 + r2, sb = b1 + b2;
    const double rho_log = lm_logavg(r1, r2, fast_rcp(r2)), b_log = lm_logavg(b1, b2, fast_rcp(b2));
    double u[D], frho[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      u[d] = avg(P1[1 + d], P2[1 + d]);
      frho[d] = u[d] * rho_log;
    }
    const double pd = fast_div(sr / 2, sb, fast_rcp(sb));
    double cc = fast_rcp(gm1x2 * b_log) - avg(P1[D + 2], P2[D + 2]) / 2;
    if (GRAV) cc = cc + avg(P1[D + 3], P2[D + 3]);
    double mv = 0;
#pragma unroll
    for (int e = 0; e < D; ++e) {
      F[1 + e] = e == R ? u[R] * frho[e] + pd : u[R] * frho[e];
      mv = e == 0 ? F[1] * u[0] : mv + F[1 + e] * u[e];
    }
    F[0] = frho[R];
    F[D + 1] = cc * frho[R] + mv;
    if (GRAV) F[1 + R] -= fast_div(sb / 2 * rho_log, 2 * b1, ib2) * (P1[D + 3] - P2[D + 3]);
  }
};

template <class L, int NQ, int SF>
ATM_DEV void fd_box_body(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q,
                         double* __restrict__ dq, double alpha, int assign, double* __restrict__ qout, double bdt,
                         int epw) {
  using PF = BoxPairEC<L>;
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA, Np = ipow(NQ, D), NP = PF::NP;
  double* sD = lds;
  double* sw = lds + NQ * NQ;
  const int tid = threadIdx.x;
  const int el = tid / Np;
  const int ijk = tid - el * Np;
  const uint32_t le = (uint32_t)blk * epw + el;  // position in the processing order
  const bool active = el < epw && le < (uint32_t)p.K;
  const uint32_t e = (p.sched && active) ? (uint32_t)p.sched[le] : le;
  double* sP = lds + NQ * NQ + NQ + el * ((NP + 1) * Np);  // [k][node], then MJ
  for (int t = tid; t < NQ * NQ; t += blockDim.x) sD[t] = p.D[t];
  for (int t = tid; t < NQ; t += blockDim.x) sw[t] = p.bw[t];
  double q1[Ns], a1[NA], P1[NP];
  const uint32_t e0 = active ? e : 0;  // a lane past the last element reads element 0 and discards it
  const uint32_t node = 8 * (e0 * Np + ijk);
  int idx[3];
  node_index<D>(ijk, NQ, idx);
  const BoxElem<D> b = *box_elem<D>(p, e0);
#pragma unroll
  for (int s = 0; s < Ns; ++s) q1[s] = ldo(p, q, s, node);
  box_aux<L>(p, node, a1);
  const double MJn = p.bw[NQ + ijk] * b.J;
  PF::prim(p.c, q1, a1, P1);
  if (active) {
#pragma unroll
    for (int k = 0; k < NP; ++k) sP[k * Np + ijk] = P1[k];
    sP[NP * Np + ijk] = MJn;
  }
  __syncthreads();
  if (!active) return;
  const double MJIn = fast_rcp(MJn);
  const double gm1x2 = 2 * (p.c.gamma - 1);
  const double ib2 = fast_rcp(2 * P1[D + 1]);
  double acc[Ns];
#pragma unroll
  for (int s = 0; s < Ns; ++s) acc[s] = assign ? 0.0 : alpha * ldo(p, dq, s, node);
  for_dirs<0, D>([&](auto R) {
    constexpr int r = decltype(R)::value, st = line_stride<NQ, r>();
    const int id = idx[r];
    const double* line = sP + ijk - id * st;
    double dl[Ns];
#pragma unroll
    for (int s = 0; s < Ns; ++s) dl[s] = -0.0;
    L::sources(p.c, dl, q1, a1, 1 << r, false);
    const double lgi = MJn * b.g[r];
#pragma unroll 1
    for (int n = 0; n < NQ; ++n) {
      double P2[NP], F[Ns];
#pragma unroll
      for (int k = 0; k < NP; ++k) P2[k] = line[k * Np + n * st];
      PF::template pair<r>(gm1x2, P1, ib2, P2, F);
      const double ci = MJIn * sD[id + NQ * n] * lgi;
      const double lgn = line[NP * Np + n * st] * b.g[r];
      const double cn = MJIn * sD[n + NQ * id];
#pragma unroll
      for (int s = 0; s < Ns; ++s) {
        dl[s] -= ci * F[s];
        dl[s] += F[s] * lgn * cn;
      }
    }
#pragma unroll
    for (int s = 0; s < Ns; ++s) acc[s] = r == 0 && assign ? dl[s] : acc[s] + dl[s];
  });
  for_dirs<0, D>([&](auto R) {
    constexpr int r = decltype(R)::value;
    const int ir = idx[r];
    if (ir != 0 && ir != NQ - 1) return;
    const bool hi = ir != 0;
    const int nb = hi ? b.nb[2 * r + 1] : b.nb[2 * r];
    constexpr int span = (NQ - 1) * line_stride<NQ, r>();
    // a boundary node reads its own state as the neighbour's and replaces it by the boundary state
    const uint32_t idp = 8 * (nb >= 0 ? (uint32_t)nb * Np + ijk + (hi ? -span : span) : e * Np + ijk);
    double qp[Ns], ap[NA], nf[Ns];
#pragma unroll
    for (int s = 0; s < Ns; ++s) qp[s] = ldo(p, q, s, idp);
    box_aux<L>(p, idp, ap);
    const double sg = hi ? 1.0 : -1.0;
    if (nb < 0) {
      double n[D];
#pragma unroll
      for (int d = 0; d < D; ++d) n[d] = d == r ? sg : 0.0;
      boundarystate<L>(p.c, n, q1, -nb, qp);
#pragma unroll
      for (int s = 0; s < NA; ++s) ap[s] = a1[s];
    }
    axis_ref_flux<L, SF, r>(p.c, sg, q1, a1, qp, ap, nf);
    double wf = 1.0;
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d != r) wf = wf * sw[idx[d]];
    const double fMJ = wf * b.fJ[r];
#pragma unroll
    for (int s = 0; s < Ns; ++s) acc[s] -= fMJ * nf[s] * MJIn;
  });
  box_epilogue<L>(p, node, q1, acc, dq, qout, bdt);
}

ATM_KERNEL_PAIR(fd_box_kernel, fd_box_body, class L ATM_COMMA int NQ ATM_COMMA int SF, L ATM_COMMA NQ ATM_COMMA SF)

template <class L, int NQ, int SF>
hipError_t launch_fd_box(const DevDG& p, hipStream_t st, const double* q, double* dq, double alpha, int assign,
                         double* qout, double bdt) {
  const int threads = ((p.epw * p.Np + 63) / 64) * 64;
  if (p.epw < 1 || threads > 512) return hipErrorInvalidConfiguration;
  const int blocks = (p.K + p.epw - 1) / p.epw;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((fd_box_kernel<L, NQ, SF>), dim3(blocks), dim3(threads), p.lds, st, p, q, dq, alpha, assign, qout,
                     bdt, p.epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF>
hipError_t launch_fd_box_batch(const BatchEntry* tab, int n, int64_t blocks, int threads, size_t lds, int epw,
                               hipStream_t st, int parity, double alpha, int assign, double b) {
  hipLaunchKernelGGL((fd_box_kernel_batch<L, NQ, SF>), dim3(blocks), dim3(threads), lds, st, tab, n, parity, alpha,
                     assign, b, epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF>
Resolved make_fd_box() {
  constexpr int Np = ipow(NQ, L::D);
  return make_resolved(launch_fd_box<L, NQ, SF>, launch_fd_box_batch<L, NQ, SF>, L::Ns, elements_per_workgroup(Np),
                       sizeof(double) * (NQ * NQ + NQ), sizeof(double) * (BoxPairEC<L>::NP + 1) * Np);
}

template <class L, int SF>
Resolved fd_box_nq(int Nq) {
  switch (Nq) {
    case 2: return make_fd_box<L, 2, SF>();
    case 3: return make_fd_box<L, 3, SF>();
    case 4: return make_fd_box<L, 4, SF>();
    case 5: return make_fd_box<L, 5, SF>();
    case 6: return make_fd_box<L, 6, SF>();
    case 7: return make_fd_box<L, 7, SF>();
    case 8: return make_fd_box<L, 8, SF>();
    default: return Resolved{nullptr, 0, 0, nullptr, 1};
  }
}

template <template <int> class LAW, int SF>
Resolved fd_box_dims(int dim, int Nq) {
  if (dim == 1) return fd_box_nq<LAW<1>, SF>(Nq);
  if (dim == 2) return fd_box_nq<LAW<2>, SF>(Nq);
  return fd_box_nq<LAW<3>, SF>(Nq);
}

}  // namespace atm
