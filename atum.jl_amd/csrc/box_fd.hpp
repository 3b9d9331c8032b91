// Entropy-conservative flux differencing in the reference's :per_dir order (src/dgsem.jl:470-561) on box
// elements: fd_body with the compact geometry.
//
// The sums keep the reference's order, every product and sum rounded; with a diagonal metric only row
// r of the two-point flux enters direction r, a third of the products.  Quotients and square roots are
// fast_div and fast_sqrt, which round as IEEE's do, by reciprocals that the pair's or node's quotients
// share; the logarithm of the logarithmic means is lm_logavg2's (a seventh of the instructions of
// the library's, and as close).  Every value equals the general kernels' but for the last bit of
// that logarithm.
//
// Bound by FP64 instructions: about 165 for an ordered pair and 290 for a face.  Against the general
// kernels, per stage: bubble 12^3 N = 4 (Roe) 78 -> 38 us, vortex 8^2 N = 4 15.5 -> 8.1 us.
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
    double rho_log, b_log;
    lm_logavg2(r1, r2, b1, b2, &rho_log, &b_log);
    const double den = gm1x2 * b_log, ii = rcp_div(sb * den);
    double u[D], frho[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      u[d] = avg(P1[1 + d], P2[1 + d]);
      frho[d] = u[d] * rho_log;
    }
    const double pd = fast_div(sr / 2, sb, den * ii);
    double cc = fast_div(1.0, den, sb * ii) - avg(P1[D + 2], P2[D + 2]) / 2;
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

// Direction r's volume sum of one node, from -0.0 on with its sources, n ascending
template <class L, int NQ, int r>
ATM_DEV void fd_box_dir(const DevDG& p, const double* sD, const double* sP, int ijk, int id, double g, double MJn,
                        double MJIn, const double* q1, const double* a1, const double* P1, double* dl) {
  using PF = BoxPairEC<L>;
  constexpr int Ns = L::Ns, Np = ipow(NQ, L::D), NP = PF::NP, st = line_stride<NQ, r>();
  const double gm1x2 = 2 * (p.c.gamma - 1);
  const double ib2 = fast_rcp(2 * P1[L::D + 1]);
  const double* line = sP + ijk - id * st;
#pragma unroll
  for (int s = 0; s < Ns; ++s) dl[s] = -0.0;
  L::sources(p.c, dl, q1, a1, 1 << r, false);
  const double lgi = MJn * g;
  // not unrolled: two pairs at once take 200 registers and gain nothing (the branch to the far
  // logarithms keeps them apart)
#pragma unroll 1
  for (int n = 0; n < NQ; ++n) {
    double P2[NP], F[Ns];
#pragma unroll
    for (int k = 0; k < NP; ++k) P2[k] = line[k * Np + n * st];
    PF::template pair<r>(gm1x2, P1, ib2, P2, F);
    const double ci = MJIn * sD[id + NQ * n] * lgi;
    const double lgn = line[NP * Np + n * st] * g;
    const double cn = MJIn * sD[n + NQ * id];
#pragma unroll
    for (int s = 0; s < Ns; ++s) {
      dl[s] -= ci * F[s];
      dl[s] += F[s] * lgn * cn;
    }
  }
}

// Byte offset of the node across the face that a node of line position ir lies on in direction r (its own
// at a boundary, so that the loads there need no branch)
template <int NQ, int D>
ATM_DEV uint32_t across(int r, bool hi, int nb, uint32_t e, int ijk) {
  const int span = (NQ - 1) * (r == 0 ? 1 : (r == 1 ? NQ : NQ * NQ));
  return 8 * (nb >= 0 ? (uint32_t)nb * ipow(NQ, D) + ijk + (hi ? -span : span) : e * ipow(NQ, D) + ijk);
}

// What the face of direction r (the outward normal sg e_r) takes from the node, qp and ap the state and
// aux across it
template <class L, int SF, int r>
ATM_DEV void fd_box_face(const DevDG& p, int nb, double sg, const double* q1, const double* a1, double* qp, double* ap,
                         double fMJ, double MJIn, double* sf) {
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA;
  if (nb < 0) {
    double n[D];
#pragma unroll
    for (int d = 0; d < D; ++d) n[d] = d == r ? sg : 0.0;
    boundarystate<L>(p.c, n, q1, -nb, qp);
#pragma unroll
    for (int s = 0; s < NA; ++s) ap[s] = a1[s];
  }
  double nf[Ns];
  axis_ref_flux<L, SF, r>(p.c, sg, q1, a1, qp, ap, nf);
#pragma unroll
  for (int s = 0; s < Ns; ++s) sf[s] = fMJ * nf[s] * MJIn;
}

// The weights' product on a face of direction r, in the order faceMJ has it
template <int D>
ATM_DEV double face_weight(const double* sw, const int idx[3], int r) {
  double wf = 1.0;
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d != r) wf = wf * sw[idx[d]];
  return wf;
}

// One thread per node: the directions one after the other.
template <class L, int NQ, int SF, class EP>
ATM_DEV void fd_box_node(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep, int epw) {
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
  const BoxElem<D>* rec = box_elem<D>(p, e0);
#pragma unroll
  for (int s = 0; s < Ns; ++s) q1[s] = ldo(p, q, s, node);
  box_aux<L>(p, node, a1);
  const double MJn = p.bw[NQ + ijk] * rec->J;
  PF::prim(p.c, q1, a1, P1);
  if (active) {
#pragma unroll
    for (int k = 0; k < NP; ++k) sP[k * Np + ijk] = P1[k];
    sP[NP * Np + ijk] = MJn;
  }
  __syncthreads();
  if (!active) return;
  const double MJIn = fast_rcp(MJn);
  double acc[Ns];
  ep.load(p, node);
  for_dirs<0, D>([&](auto R) {
    constexpr int r = decltype(R)::value;
    double dl[Ns];
    fd_box_dir<L, NQ, r>(p, sD, sP, ijk, idx[r], rec->g[r], MJn, MJIn, q1, a1, P1, dl);
#pragma unroll
    for (int s = 0; s < Ns; ++s) {
      acc[s] = r == 0 ? ep.start(s, dl[s]) : acc[s] + dl[s];
      asm("" : "+v"(acc[s]));  // summed here: the compiler would keep every direction's dl until the end
    }
  });
  for_dirs<0, D>([&](auto R) {
    constexpr int r = decltype(R)::value;
    const bool hi = idx[r] != 0;
    if (hi && idx[r] != NQ - 1) return;
    const int nb = rec->nb[2 * r + (hi ? 1 : 0)];
    const uint32_t idp = across<NQ, D>(r, hi, nb, e, ijk);
    double qp[Ns], ap[NA], sf[Ns];
#pragma unroll
    for (int s = 0; s < Ns; ++s) qp[s] = ldo(p, q, s, idp);
    box_aux<L>(p, idp, ap);
    fd_box_face<L, SF, r>(p, nb, hi ? 1.0 : -1.0, q1, a1, qp, ap, face_weight<D>(sw, idx, r) * rec->fJ[r], MJIn, sf);
#pragma unroll
    for (int s = 0; s < Ns; ++s) acc[s] -= sf[s];
  });
  ep.store(p, node, q1, acc);
}

template <class L, int NQ, int SF>
ATM_DEV void fd_box_body(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q,
                         double* __restrict__ dq, double alpha, int assign, double* __restrict__ qout, double bdt,
                         int epw) {
  StageEnd<L> ep(dq, alpha, assign, qout, bdt);
  fd_box_node<L, NQ, SF>(p, lds, blk, q, ep, epw);
}

template <class L, int NQ, int SF>
struct FdBoxBody {
  template <class EP>
  ATM_DEV static void run(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep, int epw) {
    fd_box_node<L, NQ, SF>(p, lds, blk, q, ep, epw);
  }
};

template <class L, int NQ, int SF>
__global__ void __launch_bounds__(512)
    fd_box_ark_kernel(const DevDG p, const DevDG pl, const double* __restrict__ q, const ArkSums a, int epw) {
  extern __shared__ double lds[];
  box_ark_pair<L, NQ, FdBoxBody<L, NQ, SF>>(p, pl, lds, q, a, epw);
}

// One thread per node and direction: the waves of group r (blockDim / D threads) form direction r's volume
// sum and face, and group 0 adds them up in the order above.  The same numbers; a node's chain of
// pairs, which is all the time a small mesh takes, is D times shorter.
template <class L, int NQ, int SF>
ATM_DEV void fd_box_dirs_body(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q,
                              double* __restrict__ dq, double alpha, int assign, double* __restrict__ qout, double bdt,
                              int epw) {
  using PF = BoxPairEC<L>;
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA, Np = ipow(NQ, D), NP = PF::NP;
  constexpr int stride = (NP + 1 + 2 * (D - 1) * Ns) * Np;
  double* sD = lds;
  double* sw = lds + NQ * NQ;
  const int group = blockDim.x / D;
  const int r = __builtin_amdgcn_readfirstlane(threadIdx.x / group);  // whole waves
  const int tid = threadIdx.x - r * group;
  const int el = tid / Np;
  const int ijk = tid - el * Np;
  const uint32_t le = (uint32_t)blk * epw + el;  // position in the processing order
  const bool active = el < epw && le < (uint32_t)p.K;
  const uint32_t e = (p.sched && active) ? (uint32_t)p.sched[le] : le;
  double* sP = lds + NQ * NQ + NQ + el * stride;  // [k][node], MJ, then [r - 1][volume, face][s][node]
  double* sx = sP + (NP + 1) * Np;
  for (int t = threadIdx.x; t < NQ * NQ; t += blockDim.x) sD[t] = p.D[t];
  for (int t = threadIdx.x; t < NQ; t += blockDim.x) sw[t] = p.bw[t];
  double q1[Ns], a1[NA], P1[NP], qp[Ns], ap[NA], dq0[Ns];
  const uint32_t e0 = active ? e : 0;  // a lane past the last element reads element 0 and discards it
  const uint32_t node = 8 * (e0 * Np + ijk);
  int idx[3];
  node_index<D>(ijk, NQ, idx);
  const BoxElem<D>* rec = box_elem<D>(p, e0);
  const int ir = r == 0 ? idx[0] : (r == 1 ? idx[1] : idx[2]);
  const bool hi = ir != 0, face = ir == 0 || ir == NQ - 1;
  const int nb = rec->nb[2 * r + (hi ? 1 : 0)];
#pragma unroll
  for (int s = 0; s < Ns; ++s) q1[s] = ldo(p, q, s, node);
  box_aux<L>(p, node, a1);
  const double MJn = p.bw[NQ + ijk] * rec->J, g = rec->g[r], fJ = rec->fJ[r];
  // a node inside the element reads itself
  const uint32_t idp = face ? across<NQ, D>(r, hi, nb, e0, ijk) : node;
#pragma unroll
  for (int s = 0; s < Ns; ++s) qp[s] = ldo(p, q, s, idp);
  box_aux<L>(p, idp, ap);
#pragma unroll
  for (int s = 0; s < Ns; ++s) dq0[s] = assign || r > 0 ? 0.0 : ldo(p, dq, s, node);
  if (r == 0) {
    PF::prim(p.c, q1, a1, P1);
    if (active) {
#pragma unroll
      for (int k = 0; k < NP; ++k) sP[k * Np + ijk] = P1[k];
      sP[NP * Np + ijk] = MJn;
    }
  }
  __syncthreads();
  const double MJIn = fast_rcp(MJn);
  double dl[Ns], sf[Ns];
  if (active) {
#pragma unroll
    for (int k = 0; k < NP; ++k) P1[k] = sP[k * Np + ijk];
    const double fMJ = face_weight<D>(sw, idx, r) * fJ, sg = hi ? 1.0 : -1.0;
    for_dirs<0, D>([&](auto R) {
      constexpr int rc = decltype(R)::value;
      if (r != rc) return;
      fd_box_dir<L, NQ, rc>(p, sD, sP, ijk, ir, g, MJn, MJIn, q1, a1, P1, dl);
      if (face) fd_box_face<L, SF, rc>(p, nb, sg, q1, a1, qp, ap, fMJ, MJIn, sf);
    });
    if (r > 0) {
      double* x = sx + (r - 1) * (2 * Ns * Np) + ijk;
#pragma unroll
      for (int s = 0; s < Ns; ++s) x[s * Np] = dl[s];
      if (face) {
#pragma unroll
        for (int s = 0; s < Ns; ++s) x[(Ns + s) * Np] = sf[s];
      }
    }
  }
  __syncthreads();
  if (!active || r > 0) return;
  double acc[Ns];
#pragma unroll
  for (int s = 0; s < Ns; ++s) {
    acc[s] = assign ? dl[s] : alpha * dq0[s] + dl[s];
#pragma unroll
    for (int d = 1; d < D; ++d) acc[s] = acc[s] + sx[((d - 1) * 2 * Ns + s) * Np + ijk];
    if (face) acc[s] -= sf[s];
#pragma unroll
    for (int d = 1; d < D; ++d)
      if (idx[d] == 0 || idx[d] == NQ - 1) acc[s] -= sx[((d - 1) * 2 * Ns + Ns + s) * Np + ijk];
  }
  box_epilogue<L>(p, node, q1, acc, dq, qout, bdt);
}

// Workgroups of the form that deals a line's pairs out: twelve waves leave each 168 registers
constexpr int FD_PAIRS_THREADS = 768;

// The pairs of a line dealt out too: group (r, g) forms direction r's pairs with the partners n = g, g + G, ...
// and leaves their fluxes in LDS; group (r, 0) then adds them up in the order of fd_box_dir while the last one,
// (r, G - 1), forms the face, and group (0, 0) puts the directions together.  The same numbers.  Without DEAL
// there is one group a direction, which adds its pairs up as it forms them.  A small mesh
// is bound by one node's chain of pairs (128 waves, bubble 4^3 N = 4, take 14 us a stage, 9 cycles an
// instruction), which this makes G times shorter.
template <class L, int NQ, bool DEAL>
struct FdPairs {
  static constexpr int D = L::D, Ns = L::Ns, Np = ipow(NQ, D), NP = BoxPairEC<L>::NP;
  static constexpr int NF = DEAL ? D * NQ * Ns : 0;  // flux planes, [r][n][s]
  // planes: primitives, MJ, fluxes, then [r][volume, face][s]
  static constexpr int stride = (NP + 1 + NF + 2 * D * Ns) * Np;
  // groups of partners for workgroups of `threads` per group (1: none)
  static constexpr int groups(int threads) {
    const int g = FD_PAIRS_THREADS / (D * threads);
    return g > NQ ? NQ : g;
  }
  static constexpr size_t lds(int epw) { return sizeof(double) * (size_t)(NQ * NQ + NQ + epw * stride); }
};

template <class L, int NQ, int SF, bool DEAL, class EP>
ATM_DEV void fd_box_pairs_node(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep, int epw,
                               int group) {
  using PF = BoxPairEC<L>;
  using S = FdPairs<L, NQ, DEAL>;
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA, Np = S::Np, NP = S::NP;
  double* sD = lds;
  double* sw = lds + NQ * NQ;
  const int G = DEAL ? blockDim.x / (D * group) : 1;
  const int rg = __builtin_amdgcn_readfirstlane(threadIdx.x / group);  // whole waves
  const int r = rg / G, gr = rg - r * G;
  const int tid = threadIdx.x - rg * group;
  const int el = tid / Np;
  const int ijk = tid - el * Np;
  const uint32_t le = (uint32_t)blk * epw + el;  // position in the processing order
  const bool active = el < epw && le < (uint32_t)p.K;
  const uint32_t e = (p.sched && active) ? (uint32_t)p.sched[le] : le;
  // a lane past the last element reads element 0 and discards it; its LDS is never written
  double* sP = lds + NQ * NQ + NQ + (active ? el : 0) * S::stride;
  double* sF = sP + (NP + 1) * Np;
  double* sx = sF + S::NF * Np;
  for (int t = threadIdx.x; t < NQ * NQ; t += blockDim.x) sD[t] = p.D[t];
  for (int t = threadIdx.x; t < NQ; t += blockDim.x) sw[t] = p.bw[t];
  double q1[Ns], a1[NA], qp[Ns], ap[NA];
  const uint32_t e0 = active ? e : 0;
  const uint32_t node = 8 * (e0 * Np + ijk);
  int idx[3];
  node_index<D>(ijk, NQ, idx);
  const BoxElem<D>* rec = box_elem<D>(p, e0);
  const int ir = r == 0 ? idx[0] : (r == 1 ? idx[1] : idx[2]);
  const bool hi = ir != 0, face = (ir == 0 || ir == NQ - 1) && gr == G - 1;
  const int nb = rec->nb[2 * r + (hi ? 1 : 0)];
#pragma unroll
  for (int s = 0; s < Ns; ++s) q1[s] = ldo(p, q, s, node);
  box_aux<L>(p, node, a1);
  const double MJn = p.bw[NQ + ijk] * rec->J, g = rec->g[r], fJ = rec->fJ[r];
  // a node inside the element, or of a group that takes no face, reads itself
  const uint32_t idp = face ? across<NQ, D>(r, hi, nb, e0, ijk) : node;
#pragma unroll
  for (int s = 0; s < Ns; ++s) qp[s] = ldo(p, q, s, idp);
  box_aux<L>(p, idp, ap);
  if (rg == 0) {
    ep.load(p, node);
    double P1[NP];
    PF::prim(p.c, q1, a1, P1);
    if (active) {
#pragma unroll
      for (int k = 0; k < NP; ++k) sP[k * Np + ijk] = P1[k];
      sP[NP * Np + ijk] = MJn;
    }
  }
  __syncthreads();
  const double MJIn = fast_rcp(MJn);
  const double gm1x2 = 2 * (p.c.gamma - 1);
  if (active) {
    double P1[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) P1[k] = sP[k * Np + ijk];
    const double ib2 = fast_rcp(2 * P1[D + 1]);
    for_dirs<0, D>([&](auto R) {
      constexpr int rc = decltype(R)::value, st = line_stride<NQ, rc>();
      if (r != rc) return;
      if constexpr (!DEAL) {
        double dl[Ns];
        fd_box_dir<L, NQ, rc>(p, sD, sP, ijk, ir, g, MJn, MJIn, q1, a1, P1, dl);
#pragma unroll
        for (int s = 0; s < Ns; ++s) sx[(2 * rc * Ns + s) * Np + ijk] = dl[s];
        return;
      }
      const double* line = sP + ijk - ir * st;
#pragma unroll 1
      for (int n = gr; n < NQ; n += G) {
        double P2[NP], F[Ns];
#pragma unroll
        for (int k = 0; k < NP; ++k) P2[k] = line[k * Np + n * st];
        PF::template pair<rc>(gm1x2, P1, ib2, P2, F);
#pragma unroll
        for (int s = 0; s < Ns; ++s) sF[((rc * NQ + n) * Ns + s) * Np + ijk] = F[s];
      }
    });
  }
  if (DEAL) __syncthreads();  // fluxes written
  if (active) {
    if (DEAL && gr == 0) {
      double dl[Ns];
#pragma unroll
      for (int s = 0; s < Ns; ++s) dl[s] = -0.0;
      for_dirs<0, D>([&](auto R) {
        constexpr int rc = decltype(R)::value;
        if (r == rc) L::sources(p.c, dl, q1, a1, 1 << rc, false);
      });
      const double lgi = MJn * g;
      const int st = r == 0 ? 1 : (r == 1 ? NQ : NQ * NQ);
      const double* mj = sP + NP * Np + ijk - ir * st;
      const double* F = sF + r * NQ * Ns * Np + ijk;
#pragma unroll 1
      for (int n = 0; n < NQ; ++n) {
        const double ci = MJIn * sD[ir + NQ * n] * lgi;
        const double lgn = mj[n * st] * g;
        const double cn = MJIn * sD[n + NQ * ir];
#pragma unroll
        for (int s = 0; s < Ns; ++s) {
          const double f = F[(n * Ns + s) * Np];
          dl[s] -= ci * f;
          dl[s] += f * lgn * cn;
        }
      }
#pragma unroll
      for (int s = 0; s < Ns; ++s) sx[(2 * r * Ns + s) * Np + ijk] = dl[s];
    }
    if (face) {
      double sf[Ns];
      const double fMJ = face_weight<D>(sw, idx, r) * fJ, sg = hi ? 1.0 : -1.0;
      for_dirs<0, D>([&](auto R) {
        constexpr int rc = decltype(R)::value;
        if (r == rc) fd_box_face<L, SF, rc>(p, nb, sg, q1, a1, qp, ap, fMJ, MJIn, sf);
      });
#pragma unroll
      for (int s = 0; s < Ns; ++s) sx[((2 * r + 1) * Ns + s) * Np + ijk] = sf[s];
    }
  }
  __syncthreads();
  if (!active || rg > 0) return;
  double acc[Ns];
#pragma unroll
  for (int s = 0; s < Ns; ++s) {
    acc[s] = ep.start(s, sx[s * Np + ijk]);
#pragma unroll
    for (int d = 1; d < D; ++d) acc[s] = acc[s] + sx[(2 * d * Ns + s) * Np + ijk];
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (idx[d] == 0 || idx[d] == NQ - 1) acc[s] -= sx[((2 * d + 1) * Ns + s) * Np + ijk];
  }
  ep.store(p, node, q1, acc);
}

// Largest workgroup of the form with a thread per node and direction: the 2-D kernels' (every shape fits).
// Per stage, one thread per node against one per node and direction: vortex 8^2 N = 4 12.2 -> 8.2 us,
// 32^2 N = 3 8.8 -> 6.8, 30^2 N = 7 14.1 -> 12.6, 64^2 N = 4 13.5 -> 13.5, 45^2 N = 6 16.9 -> 16.4.  Of a larger
// 3-D mesh its six-wave workgroups of 168 registers leave too few resident: bubble 12^3 N = 4 38 -> 57 us,
// 14^3 N = 3 26.4 -> 30.4.
template <class L>
constexpr int fd_box_dirs_threads() {
  return L::D == 2 ? 1024 : 0;
}

template <class L, int NQ>
constexpr size_t fd_box_elem_bytes() {
  constexpr int planes = BoxPairEC<L>::NP + 1 + (fd_box_dirs_threads<L>() > 0 ? 2 * (L::D - 1) * L::Ns : 0);
  return sizeof(double) * planes * ipow(NQ, L::D);
}

template <class L, int NQ, int SF>
__global__ void __attribute__((amdgpu_flat_work_group_size(1, fd_box_dirs_threads<L>())))
fd_box_dirs_kernel(const DevDG p, const double* __restrict__ q, double* __restrict__ dq, double alpha, int assign,
                   double* __restrict__ qout, double bdt, int epw) {
  extern __shared__ double lds[];
  fd_box_dirs_body<L, NQ, SF>(p, lds, xcd_block(), q, dq, alpha, assign, qout, bdt, epw);
}

template <class L, int NQ, int SF>
__global__ void __attribute__((amdgpu_flat_work_group_size(1, fd_box_dirs_threads<L>())))
fd_box_dirs_kernel_batch(const BatchEntry* __restrict__ tab, int n, int parity, double alpha, int assign, double b,
                         int epw) {
  extern __shared__ double lds[];
  const int64_t lb = xcd_block();
  const int i = batch_find(tab, n, lb);
  const DevDG p = tab[i].p;
  fd_box_dirs_body<L, NQ, SF>(p, lds, lb - tab[i].block_start, tab[i].buf[parity], tab[i].dq, alpha, assign,
                              tab[i].buf[1 - parity], b * tab[i].dt, epw);
}

template <class L, int NQ, int SF, bool DEAL>
__global__ void __launch_bounds__(FD_PAIRS_THREADS)
    fd_box_pairs_kernel(const DevDG p, const double* __restrict__ q, double* __restrict__ dq, double alpha, int assign,
                        double* __restrict__ qout, double bdt, int epw, int group) {
  extern __shared__ double lds[];
  StageEnd<L> ep(dq, alpha, assign, qout, bdt);
  fd_box_pairs_node<L, NQ, SF, DEAL>(p, lds, xcd_block(), q, ep, epw, group);
}

// Whether a mesh's pairs are dealt out over groups of threads: where every CU has one workgroup at most.  Per
// pass of two LSRK54 steps, against a thread per node and direction (2-D) or per node (3-D), with up to 256
// workgroups: vortex 8^2 N = 4 78 -> 66 us, 16^2 N = 4 74 -> 66, 16^2 N = 7 96 -> 75, 32^2 N = 3 63 -> 60,
// bubble 6^3 N = 4 146 -> 113, 5^3 N = 3 120 -> 91, 12^3 N = 1 87 -> 69; with more: vortex 24^2 N = 4 83 -> 97,
// 20^2 N = 6 103 -> 113, bubble 7^3 N = 4 208 -> 206, 7^3 N = 3 125 -> 163.
constexpr int FD_PAIRS_BLOCKS = 256;
// In 3-D up to two workgroups a CU and a wave per SIMD the directions alone are dealt out.  Per pass, a thread per
// node against one per node and direction: bubble 7^3 N = 3 123 -> 100 us, 8^3 N = 4 207 -> 189, 9^3 N = 2
// 114 -> 94, 6^3 N = 5 166 -> 156, 14^3 N = 1 93 -> 79, two ARK23 steps on 8x8x6 N = 3 137 -> 123; beyond:
// 10^3 N = 3 132 -> 131, 12^3 N = 2 121 -> 122, 20^3 N = 1 102 -> 105, 11x11x7 157 -> 156.
constexpr int FD_DIRS_BLOCKS = 512, FD_DIRS_WAVES = 1024;
// Calls f(DEAL, groups of partners, LDS) if a launch takes that form
template <class L, int NQ, class F>
bool fd_box_dealt(const DevDG& p, int blocks, int threads, F&& f) {
  if (p.epw < 1 || blocks < 1) return false;
  const int G = FdPairs<L, NQ, true>::groups(threads);
  const size_t lds = FdPairs<L, NQ, true>::lds(p.epw);
  if (blocks <= FD_PAIRS_BLOCKS && G > 1 && lds <= 160 * 1024) {
    f(std::true_type{}, G, lds);
    return true;
  }
  if constexpr (L::D == 3) {
    const size_t lds1 = FdPairs<L, NQ, false>::lds(p.epw);
    if (L::D * threads <= FD_PAIRS_THREADS && blocks <= FD_DIRS_BLOCKS &&
        (int64_t)blocks * threads <= 64 * FD_DIRS_WAVES && lds1 <= 160 * 1024) {
      f(std::false_type{}, 1, lds1);
      return true;
    }
  }
  return false;
}

template <class L, int NQ, int SF, bool DEAL>
struct FdPairsBody {
  template <class EP>
  ATM_DEV static void run(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep, int epw) {
    fd_box_pairs_node<L, NQ, SF, DEAL>(p, lds, blk, q, ep, epw, (epw * ipow(NQ, L::D) + 63) / 64 * 64);
  }
};

template <class L, int NQ, int SF, bool DEAL>
__global__ void __launch_bounds__(FD_PAIRS_THREADS)
    fd_box_pairs_ark_kernel(const DevDG p, const DevDG pl, const double* __restrict__ q, const ArkSums a, int epw) {
  extern __shared__ double lds[];
  box_ark_pair<L, NQ, FdPairsBody<L, NQ, SF, DEAL>>(p, pl, lds, q, a, epw);
}

template <class L, int NQ, int SF>
hipError_t launch_fd_box_ark(const DevDG& p, const DevDG& pl, hipStream_t st, const double* q, const ArkSums& a) {
  const int threads = ((p.epw * p.Np + 63) / 64) * 64, blocks = p.epw < 1 ? 0 : (p.K + p.epw - 1) / p.epw;
  // (an element's planes of the explicit form outnumber the implicit one's)
  if (fd_box_dealt<L, NQ>(p, blocks, threads, [&](auto deal, int G, size_t lds) {
        constexpr bool DEAL = decltype(deal)::value;
        hipLaunchKernelGGL((fd_box_pairs_ark_kernel<L, NQ, SF, DEAL>), dim3(blocks), dim3(L::D * G * threads), lds, st, p,
                           pl, q, a, p.epw);
      }))
    return hipGetLastError();
  return launch_box_ark_pair<L, NQ>(fd_box_ark_kernel<L, NQ, SF>, 512, p, pl, st, q, a);
}

ATM_KERNEL_PAIR(fd_box_kernel, fd_box_body, class L ATM_COMMA int NQ ATM_COMMA int SF, L ATM_COMMA NQ ATM_COMMA SF)

template <class L, int NQ, int SF>
hipError_t launch_fd_box(const DevDG& p, hipStream_t st, const double* q, double* dq, double alpha, int assign,
                         double* qout, double bdt) {
  const int threads = ((p.epw * p.Np + 63) / 64) * 64;
  if (p.epw < 1 || threads > 512) return hipErrorInvalidConfiguration;
  const int blocks = (p.K + p.epw - 1) / p.epw;
  if (blocks == 0) return hipSuccess;
  if constexpr (L::D > 1)
    if (fd_box_dealt<L, NQ>(p, blocks, threads, [&](auto deal, int G, size_t lds) {
          constexpr bool DEAL = decltype(deal)::value;
          hipLaunchKernelGGL((fd_box_pairs_kernel<L, NQ, SF, DEAL>), dim3(blocks), dim3(L::D * G * threads), lds, st, p,
                             q, dq, alpha, assign, qout, bdt, p.epw, threads);
        }))
      return hipGetLastError();
  if constexpr (fd_box_dirs_threads<L>() > 0)
    if (L::D * threads <= fd_box_dirs_threads<L>()) {
      hipLaunchKernelGGL((fd_box_dirs_kernel<L, NQ, SF>), dim3(blocks), dim3(L::D * threads), p.lds, st, p, q, dq,
                         alpha, assign, qout, bdt, p.epw);
      return hipGetLastError();
    }
  hipLaunchKernelGGL((fd_box_kernel<L, NQ, SF>), dim3(blocks), dim3(threads), p.lds, st, p, q, dq, alpha, assign, qout,
                     bdt, p.epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF>
hipError_t launch_fd_box_batch(const BatchEntry* tab, int n, int64_t blocks, int threads, size_t lds, int epw,
                               hipStream_t st, int parity, double alpha, int assign, double b) {
  if constexpr (fd_box_dirs_threads<L>() > 0)
    if (L::D * threads <= fd_box_dirs_threads<L>()) {
      hipLaunchKernelGGL((fd_box_dirs_kernel_batch<L, NQ, SF>), dim3(blocks), dim3(L::D * threads), lds, st, tab, n,
                         parity, alpha, assign, b, epw);
      return hipGetLastError();
    }
  hipLaunchKernelGGL((fd_box_kernel_batch<L, NQ, SF>), dim3(blocks), dim3(threads), lds, st, tab, n, parity, alpha,
                     assign, b, epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF>
Resolved make_fd_box() {
  constexpr int Np = ipow(NQ, L::D);
  // one wave of small elements by default, as the FAST kernels
  Resolved r = make_resolved(launch_fd_box<L, NQ, SF>, launch_fd_box_batch<L, NQ, SF>, L::Ns, Np >= 64 ? 1 : 64 / Np,
                             sizeof(double) * (NQ * NQ + NQ), fd_box_elem_bytes<L, NQ>());
  if constexpr (L::LAW == ATM_LAW_EULER_GRAVITY && L::D == 3) r.pfn = launch_fd_box_ark<L, NQ, SF>;
  return r;
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
