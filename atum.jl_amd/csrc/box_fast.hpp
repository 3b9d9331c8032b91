// Pair-symmetric EC flux-differencing kernel (ATM_PRECISION_FAST) on box elements.
//
// The operator of fd_fast.hpp with the geometry of a box taken out of the sums.  With a diagonal
// metric and MJ = J w_i w_j w_k a pair {a, b} of a line in direction r has
//   MJI_a G_ab = (g_r / w_a) S_ab,   S_ab = D[b,a] w_b - D[a,b] w_a = -S_ba,
// so a node needs only row r of the two-point flux, one table entry per pair and one factor per
// direction; MJ, MJI and the metric rows are not read at all.  The surface term scales as
// faceMJ MJI = g_r / w_end.  A face's flux is evaluated in a frame turned (and for the low face
// reflected) so that the outward normal is the first axis: the normal's zeros and ones drop out.
//
// Work split as in fd_fast.hpp: thread = node, tournament pairing, the partner's share through LDS.
// The shares of at most SLOTS pair distances are exchanged at a time, which bounds the element's LDS
// for the high degrees.
#pragma once
#include "box.hpp"
#include "fd_fast.hpp"
#include "log_mean.hpp"

namespace atm {

// Pair distances exchanged in one round
constexpr int BOX_SLOTS = 2;

template <class L, int NQ>
constexpr int box_xbuf() {
  constexpr int D = L::D, Ns = L::Ns, Np = ipow(NQ, D), M = NQ / 2;
  // a round of BOX_SLOTS distances, or all of them; with even NQ the last distance has half the shares
  constexpr int full = M <= BOX_SLOTS ? (NQ % 2 == 0 ? (M - 1) * Ns * Np + Ns * (Np / 2) : M * Ns * Np)
                                      : BOX_SLOTS * Ns * Np;
  constexpr int faces = 2 * D * (Np / NQ) * Ns;
  return full > faces ? full : faces;
}

// Entropy-conservative two-point flux of the Euler laws from per-node primitives
// [rho, u/2 (D), b = rho/2p, phi/2 (gravity), 1/2b (gravity)]: row r of twice the flux.  With
// rl = 2 rho_log, pd = 2 rho_avg / 2 b_avg and u the pair average,
//   F_r = [rl u_r, rl u_r u + pd e_r, u_r (rl (1/(2 (gamma-1) b_log) + phi_avg + u_a.u_b/2) + pd)]
// (|u|^2 - |u|^2_avg/2 of the reference's energy flux is u_a.u_b/2), and the gravity fluctuation of node
// a takes t / 2b_a, t = 2 b_avg rl (phi_a - phi_b)/2, from its momentum.  Halved velocities and potentials
// and the factor 2, which the table S_ab takes back, save the multiplications by 1/2 in every mean.
template <class L>
struct BoxEC {
  static constexpr int D = L::D, Ns = L::Ns;
  static constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  static constexpr int NP = GRAV ? D + 4 : D + 2;  // LDS planes
  ATM_DEV static void prim(const LawConst& c, const double* q, double phi, double* P) {
#pragma clang fp contract(fast)
    const double ir = fast_rcp(q[0]), hr = 0.5 * ir;
    double ke = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      P[1 + d] = q[1 + d] * hr;
      ke += P[1 + d] * q[1 + d];
    }
    double e = q[D + 1] - ke;
    if (GRAV) e -= q[0] * phi;
    const double ib = 2 * (c.gamma - 1) * e * ir;  // 1/b = 2p/rho
    P[0] = q[0];
    P[D + 1] = fast_rcp(ib);
    if (GRAV) {
      P[D + 2] = 0.5 * phi;
      P[D + 3] = 0.5 * ib;
    }
  }
  // sf: S/2 times row r of twice the flux's symmetric part; the fluctuation takes ta from momentum r
  // of node a's sum and adds tb to what node b subtracts
  template <int r>
  ATM_DEV static void pair(double inv_gm1, const double* Pa, const double* Pb, double S, double* sf, double* ta,
                           double* tb) {
#pragma clang fp contract(fast)
    const double ra = Pa[0], rb = Pb[0], ba = Pa[D + 1], bb = Pb[D + 1];
    const double sr = ra + rb, sb = ba + bb;
    const double i2 = fast_rcp(sr * sb);
    const double isr = sb * i2, isb = sr * i2;
    const double fr = (ra - rb) * isr, fb = (ba - bb) * isb;
    const double ur = fr * fr, ub = fb * fb;
    double Gr, Fb;
    if (ur < LM_U && ub < LM_U) {
      Gr = lm_inverse(ur);
      Fb = lm_direct(ub);
    } else {
      Gr = lm_g(ra, rb, ur);
      Fb = lm_f(ba, bb, ub);
    }
    const double rl = sr * Gr;
    const double pd = sr * isb;
    double u[D], dot = Pa[1] * Pb[1];
#pragma unroll
    for (int d = 1; d < D; ++d) dot += Pa[1 + d] * Pb[1 + d];
#pragma unroll
    for (int d = 0; d < D; ++d) u[d] = Pa[1 + d] + Pb[1 + d];
    double cc = Fb * isb * inv_gm1;
    if (GRAV) cc += Pa[D + 2] + Pb[D + 2];
    cc += 2 * dot;
    const double su = S * u[r];
    sf[0] = rl * su;
#pragma unroll
    for (int d = 0; d < D; ++d) sf[1 + d] = u[d] * sf[0];
    sf[1 + r] += pd * S;
    sf[D + 1] = su * (rl * cc + pd);
    if (GRAV) {
      const double t = S * (sb * rl * (Pa[D + 2] - Pb[D + 2]));
      *ta = t * Pa[D + 3];
      *tb = t * Pb[D + 3];
      asm("" : "+v"(*ta));
    }
    // rounded here: a kernel could otherwise fuse the last product of one into the sum it goes to and another not
#pragma unroll
    for (int s = 0; s < Ns; ++s) asm("" : "+v"(sf[s]));
  }
};

template <class L, int NQ>
constexpr size_t fast_box_elem_doubles() {
  return (size_t)BoxEC<L>::NP * ipow(NQ, L::D) + box_xbuf<L, NQ>();
}

// FAST surface flux with the normal along the first momentum component
template <class L, int SF>
ATM_DEV void axis_fast_flux(const LawConst& c, const double* qm, double phim, double prefm, const double* qp,
                            double phip, double prefp, double* nf) {
  constexpr int D = L::D, Ns = L::Ns;
  constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  // the pressures keep the reference's rounding (fast_flux.hpp): the law's pressure() with its
  // division rounded the same by fast_div
  const double irm = fast_rcp(qm[0]), irp = fast_rcp(qp[0]);
  const double gm1 = c.gamma - 1;
  const double em = qm[D + 1] - fast_div(dotv<D>(qm + 1, qm + 1), 2 * qm[0], 0.5 * irm);
  const double ep = qp[D + 1] - fast_div(dotv<D>(qp + 1, qp + 1), 2 * qp[0], 0.5 * irp);
  const double pm = gm1 * (GRAV ? em - qm[0] * phim : em);
  const double pfp = gm1 * (GRAV ? ep - qp[0] * phip : ep);
  const double pp = GRAV && SF == ATM_FLUX_ROE ? gm1 * (ep - qp[0] * phim) : pfp;
  {
#pragma clang fp contract(fast)
    double um[D], up[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      um[d] = qm[1 + d] * irm;
      up[d] = qp[1 + d] * irp;
    }
    const double unm = um[0], unp = up[0];
    // sum of the normal physical fluxes
    double fs[Ns];
    fs[0] = qm[1] + qp[1];
#pragma unroll
    for (int d = 0; d < D; ++d) fs[1 + d] = qm[1 + d] * unm + qp[1 + d] * unp;
    fs[1] += (pm - prefm) + (pfp - prefp);
    fs[D + 1] = unm * (qm[D + 1] + pm) + unp * (qp[D + 1] + pfp);
    if constexpr (SF == ATM_FLUX_RUSANOV) {
      const double wm = fabs(unm) + fast_sqrt(c.gamma * pm * irm);
      const double wp = fabs(unp) + fast_sqrt(c.gamma * pfp * irp);
      const double ws = 0.5 * fmax(wm, wp);
#pragma unroll
      for (int s = 0; s < Ns; ++s) nf[s] = 0.5 * fs[s] - ws * (qp[s] - qm[s]);
    } else {
      const double hm = (qm[D + 1] + pm) * irm, hp = (qp[D + 1] + pp) * irp;
      const double cm = fast_sqrt(c.gamma * pm * irm), cp = fast_sqrt(c.gamma * pp * irp);
      const double srm = fast_sqrt(qm[0]), srp = fast_sqrt(qp[0]);
      const double iden = fast_rcp(srm + srp);
      const double rho = srm * srp;
      double u[D], du[D], uu = 0, udu = 0;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        u[d] = (srm * um[d] + srp * up[d]) * iden;
        du[d] = up[d] - um[d];
        uu += u[d] * u[d];
        if (d > 0) udu += u[d] * du[d];  // u.du - (u.n)(du.n)
      }
      const double un = u[0], dun = du[0];
      const double h = (srm * hm + srp * hp) * iden;
      const double cs = (srm * cm + srp * cp) * iden;
      const double drho = qp[0] - qm[0], dp = pp - pm;
      const double cm2 = fast_rcp(cs * cs);
      const double w1 = 0.5 * fabs(un - cs) * (dp - rho * cs * dun) * cm2;
      const double w2 = 0.5 * fabs(un + cs) * (dp + rho * cs * dun) * cm2;
      const double w3 = fabs(un) * (drho - dp * cm2);
      const double w4 = fabs(un) * rho;
      const double e3 = GRAV ? w3 * (0.5 * uu + phim) : 0.5 * w3 * uu;
      const double ws = w1 + w2 + w3, wc = cs * (w2 - w1);
      nf[0] = 0.5 * fs[0] - 0.5 * ws;
      nf[1] = 0.5 * fs[1] - 0.5 * (ws * u[0] + wc);
#pragma unroll
      for (int d = 1; d < D; ++d) nf[1 + d] = 0.5 * fs[1 + d] - 0.5 * (ws * u[d] + w4 * du[d]);
      nf[D + 1] = 0.5 * fs[D + 1] - 0.5 * ((w1 + w2) * h + wc * un + e3 + w4 * udu);
    }
  }
}

// The face points of an element dealt out over its threads (FastFaces of fd_fast.hpp): point
// f = t + i Np in round i; buf[s * NFP + f] takes the flux times g_r / w_end.
template <class L, int SF, int NQ>
struct BoxFaces {
  static constexpr int D = L::D, Ns = L::Ns, Np = ipow(NQ, D), NFPF = Np / NQ, NFP = 2 * D * NFPF;
  static constexpr int R = (NFP + Np - 1) / Np;  // rounds
  static constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  int nb[R];  // neighbour element or minus the boundary tag
  // a round past the last face point reads the last face's entry and ignores it
  ATM_DEV void load(const BoxElem<D>* rec, int t) {
#pragma unroll
    for (int i = 0; i < R; ++i) nb[i] = rec->nb[min(t + i * Np, NFP - 1) / NFPF];
  }
  // sQ: [s][node] the element's state and, for Euler-gravity, its geopotential (s = Ns); iw: 1 / w_end
  ATM_DEV void run(const DevDG& p, const BoxElem<D>* rec, uint32_t e, int t, const double* q, double* buf,
                   const double* sQ, double iw) const {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int f = t + i * Np;
      if (f >= NFP) break;
      const int face = f / NFPF, fp = f - face * NFPF, r = face >> 1;
      const bool hi = face & 1;
      const int st = r == 0 ? 1 : (r == 1 ? NQ : NQ * NQ);
      // face point (i, j) -> node: (0, i, j), (i, 0, j) or (i, j, 0)
      const int ln0 = r == 0 ? fp * NQ : (r == 1 ? fp + (NQ * NQ - NQ) * (fp / NQ) : fp);
      const int ln = ln0 + (hi ? (NQ - 1) * st : 0);
      // a boundary face point reads its own node as the neighbour (every load unconditional)
      const uint32_t own = 8 * (e * Np + ln);
      const uint32_t idp = nb[i] >= 0 ? 8 * ((uint32_t)nb[i] * Np + ln0 + (hi ? 0 : (NQ - 1) * st)) : own;
      const uint32_t plane = 8 * (uint32_t)p.Ntot;
      const double sg = hi ? 1.0 : -1.0;
      const double lf = rec->g[r] * iw;
      int pl[D];  // state planes of the turned momentum components
#pragma unroll
      for (int d = 0; d < D; ++d) pl[d] = 1 + (r + d >= D ? r + d - D : r + d);
      double qp[Ns], qm[Ns], nf[Ns];
      qp[0] = ldo(p, q, 0, idp);
#pragma unroll
      for (int d = 0; d < D; ++d) qp[1 + d] = ldo(p, q, 0, idp + pl[d] * plane);
      qp[D + 1] = ldo(p, q, D + 1, idp);
      const double phip0 = GRAV ? ldo(p, p.aux, 0, idp) : 0.0;
      qm[0] = sQ[ln];
#pragma unroll
      for (int d = 0; d < D; ++d) qm[1 + d] = sQ[pl[d] * Np + ln];
      qm[D + 1] = sQ[(D + 1) * Np + ln];
      const double phim = GRAV ? sQ[Ns * Np + ln] : 0.0;
      double phip = phip0;
      double prefm = 0.0, prefp = 0.0;
      if (GRAV && p.c.pde_level_balance) {  // uniform over the launch
        prefm = ldo(p, p.aux, D + 2, own);
        prefp = ldo(p, p.aux, D + 2, idp);
      }
      qm[1] *= sg;
      qp[1] *= sg;
      if (nb[i] < 0) {
        phip = phim;
        prefp = prefm;
        if (p.c.bc == ATM_BC_REFLECT) {
#pragma unroll
          for (int s = 0; s < Ns; ++s) qp[s] = qm[s];
          qp[1] = qm[1] - 2 * qm[1];
        } else {
          // the other boundary states are defined in the mesh frame
          double n[D], qo[Ns], qb[Ns];
#pragma unroll
          for (int d = 0; d < D; ++d) n[d] = d == r ? sg : 0.0;
#pragma unroll
          for (int s = 0; s < Ns; ++s) qo[s] = sQ[s * Np + ln];
          boundarystate<L>(p.c, n, qo, -nb[i], qb);
          qp[0] = qb[0];
#pragma unroll
          for (int d = 0; d < D; ++d) {
            double v = qb[1];
#pragma unroll
            for (int k = 1; k < D; ++k) v = pl[d] == 1 + k ? qb[1 + k] : v;
            qp[1 + d] = v;
          }
          qp[1] *= sg;
          qp[D + 1] = qb[D + 1];
        }
      }
      axis_fast_flux<L, SF>(p.c, qm, phim, prefm, qp, phip, prefp, nf);
      nf[1] *= sg;
      buf[f] = lf * nf[0];
#pragma unroll
      for (int d = 0; d < D; ++d) buf[pl[d] * NFP + f] = lf * nf[1 + d];
      buf[(D + 1) * NFP + f] = lf * nf[D + 1];
    }
  }
  ATM_DEV static void gather(const int idx[3], const double* buf, double* acc) {
#pragma unroll
    for (int r = 0; r < D; ++r) {
      const int ir = idx[r];
      if (ir != 0 && ir != NQ - 1) continue;
      int fp = 0;
      if (D == 2) fp = (r == 0) ? idx[1] : idx[0];
      if (D == 3) fp = (r == 0) ? idx[1] + NQ * idx[2] : ((r == 1) ? idx[0] + NQ * idx[2] : idx[0] + NQ * idx[1]);
      const int f = (2 * r + (ir != 0)) * NFPF + fp;
#pragma unroll
      for (int s = 0; s < Ns; ++s) acc[s] -= buf[s * NFP + f];
    }
  }
};

template <class L, int NQ, int SF, class EP>
ATM_DEV void fast_box_node(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep, int epw) {
#pragma clang fp contract(fast)
  constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  using EC = BoxEC<L>;
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA, Np = ipow(NQ, D), M = NQ / 2, NPL = EC::NP;
  constexpr bool HALF = NQ % 2 == 0;  // the pairs at distance NQ/2 are taken by the lower half of each line
  constexpr int stride = (int)fast_box_elem_doubles<L, NQ>();
  static_assert(NPL >= Ns + (GRAV ? 1 : 0), "the surface term stages the state in the primitives' planes");
  double* sS = lds;                // S_ab / 2 at [b + NQ a]
  double* siw = lds + NQ * NQ;     // 1 / w_a
  const int tid = threadIdx.x;
  const int el = tid / Np;
  const int ijk = tid - el * Np;
  const uint32_t le = (uint32_t)blk * epw + el;  // position in the processing order
  const bool active = el < epw && le < (uint32_t)p.K;
  const uint32_t e = (p.sched && active) ? (uint32_t)p.sched[le] : le;
  double* sP = lds + NQ * NQ + NQ + el * stride;  // [k][node]
  double* sx = sP + NPL * Np;                     // [slot][s][node]
  for (int t = tid; t < NQ * NQ; t += blockDim.x) {
    const int b = t % NQ, a = t / NQ;
    sS[t] = 0.5 * (p.D[b + NQ * a] * p.bw[b] - p.D[a + NQ * b] * p.bw[a]);
  }
  for (int t = tid; t < NQ; t += blockDim.x) siw[t] = 1 / p.bw[t];
  // every load of the node's data first and unconditionally (a lane past the last element reads
  // element 0 and discards it)
  const uint32_t e0 = active ? e : 0;
  const uint32_t node = 8 * (e0 * Np + ijk);
  const BoxElem<D>* rec = box_elem<D>(p, e0);
  double q1[Ns], a1[NA], P1[NPL];
#pragma unroll
  for (int s = 0; s < Ns; ++s) q1[s] = ldo(p, q, s, node);
  box_aux<L>(p, node, a1);
  double g[D];
#pragma unroll
  for (int d = 0; d < D; ++d) g[d] = rec->g[d];
  using BF = BoxFaces<L, SF, NQ>;
  BF bf;
  bf.load(rec, ijk);
  EC::prim(p.c, q1, GRAV ? a1[0] : 0.0, P1);
  if (active) {
#pragma unroll
    for (int k = 0; k < NPL; ++k) sP[k * Np + ijk] = P1[k];
  }
  int idx[3];
  node_index<D>(ijk, NQ, idx);
  // a node of the upper half of its line in direction r, at line position c >= M, by its position there
  auto half_pos = [&](int r, int c) {
    int pos = 0, st = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      pos += (d == r ? c - M : idx[d]) * st;
      st *= d == r ? M : NQ;
    }
    return pos;
  };
  const double inv_gm1 = 1 / (p.c.gamma - 1);
  double acc[Ns];
#pragma unroll
  for (int s = 0; s < Ns; ++s) acc[s] = 0.0;
  if (active) L::sources(p.c, acc, q1, a1, all_dirs<L>(), false);
  __syncthreads();  // tables and primitives written
  for_dirs<0, D>([&](auto R) {
    constexpr int r = decltype(R)::value, st = line_stride<NQ, r>();
    const int a = idx[r];
    const int lbase = ijk - a * st;
    double vol[Ns];
#pragma unroll
    for (int s = 0; s < Ns; ++s) vol[s] = 0.0;
#pragma unroll
    for (int m0 = 1; m0 <= M; m0 += BOX_SLOTS) {
      if (r > 0 || m0 > 1) __syncthreads();  // the previous round's shares are gathered
      if (active) {
#pragma unroll
        for (int m = m0; m < m0 + BOX_SLOTS && m <= M; ++m) {
          if (HALF && m == M && a >= M) continue;
          const int b = a + m >= NQ ? a + m - NQ : a + m;
          const int ib = lbase + b * st;
          double P2[NPL];
#pragma unroll
          for (int k = 0; k < NPL; ++k) P2[k] = sP[k * Np + ib];
          double sf[Ns], ta, tb;
          EC::template pair<r>(inv_gm1, P1, P2, sS[b + NQ * a], sf, &ta, &tb);
#pragma unroll
          for (int s = 0; s < Ns; ++s) vol[s] += sf[s];
          if (GRAV) {
            vol[1 + r] -= ta;
            sf[1 + r] += tb;
          }
          // the partner's share, which it subtracts
          const bool hs = HALF && m == M;
          double* slot = sx + (m - m0) * Ns * Np + (hs ? half_pos(r, b) : ib);
          const int xs = hs ? Np / 2 : Np;
#pragma unroll
          for (int s = 0; s < Ns; ++s) slot[s * xs] = sf[s];
        }
      }
      __syncthreads();
      if (active) {
#pragma unroll
        for (int m = m0; m < m0 + BOX_SLOTS && m <= M; ++m) {
          if (HALF && m == M && a < M) continue;
          const bool hs = HALF && m == M;
          const double* slot = sx + (m - m0) * Ns * Np + (hs ? half_pos(r, a) : ijk);
          const int xs = hs ? Np / 2 : Np;
#pragma unroll
          for (int s = 0; s < Ns; ++s) vol[s] -= slot[s * xs];
        }
      }
    }
    const double gw = g[r] * siw[a];
#pragma unroll
    for (int s = 0; s < Ns; ++s) {
      acc[s] += gw * vol[s];
      asm("" : "+v"(acc[s]));  // summed here: the compiler would keep every direction's vol until the end
    }
  });
  // Surface term: no thread reads a partner's primitives any more, so the state and geopotential are
  // staged by node in their planes; the face points read their own side there, the update the state.
  double* sQ = sP;
  if (active) {
#pragma unroll
    for (int s = 0; s < Ns; ++s) sQ[s * Np + ijk] = ldo(p, q, s, node);
    if constexpr (GRAV) sQ[Ns * Np + ijk] = 2 * P1[D + 2];  // = aux[0]
  }
  __syncthreads();  // every thread has consumed its exchange slots
  if (active) bf.run(p, rec, e, ijk, q, sx, sQ, siw[0]);
  __syncthreads();
  if (!active) return;
  ep.load(p, node);
#pragma unroll
  for (int s = 0; s < Ns; ++s) q1[s] = sQ[s * Np + ijk];
#pragma unroll
  for (int s = 0; s < Ns; ++s) acc[s] = ep.start_fused(s, acc[s]);
  BF::gather(idx, sx, acc);
  ep.store(p, node, q1, acc);
}

// An element's work dealt out by role: group 0 of a workgroup's threads takes direction 0 and the update, group
// r direction r, the last group the face fluxes.  The sums in the order of fast_box_node: same bits.
template <class L, int NQ>
struct FastRoles {
  static constexpr bool GRAV = L::LAW == ATM_LAW_EULER_GRAVITY;
  static constexpr int D = L::D, Ns = L::Ns, Np = ipow(NQ, D), M = NQ / 2, NPL = BoxEC<L>::NP;
  // shares of one direction, [distance][s][node], half of the last distance's with even NQ
  static constexpr int share = NQ % 2 == 0 ? (M - 1) * Ns * Np + Ns * (Np / 2) : M * Ns * Np;
  // primitives, state and geopotential, shares, the later directions' sums, face fluxes
  static constexpr int state = NPL * Np, xch = state + (Ns + GRAV) * Np, sum = xch + D * share,
                       faces = sum + (D - 1) * Ns * Np, stride = faces + 2 * D * (Np / NQ) * Ns;
  static constexpr size_t lds(int epw) { return sizeof(double) * (size_t)(NQ * NQ + NQ + epw * stride); }
};

template <class L, int NQ, int SF, class EP>
ATM_DEV void fast_box_roles_node(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep,
                                 int epw) {
#pragma clang fp contract(fast)
  using EC = BoxEC<L>;
  using S = FastRoles<L, NQ>;
  using BF = BoxFaces<L, SF, NQ>;
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA, Np = S::Np, M = S::M, NPL = S::NPL;
  constexpr bool HALF = NQ % 2 == 0, GRAV = S::GRAV;
  double* sS = lds;             // S_ab / 2 at [b + NQ a]
  double* siw = lds + NQ * NQ;  // 1 / w_a
  const int group = blockDim.x / (D + 1);
  const int role = __builtin_amdgcn_readfirstlane(threadIdx.x / group);  // whole waves
  const int tid = threadIdx.x - role * group;
  const int el = tid / Np;
  const int ijk = tid - el * Np;
  const uint32_t le = (uint32_t)blk * epw + el;  // position in the processing order
  const bool active = el < epw && le < (uint32_t)p.K;
  const uint32_t e = (p.sched && active) ? (uint32_t)p.sched[le] : le;
  // a lane past the last element reads element 0 and writes nothing
  double* sP = lds + NQ * NQ + NQ + (active ? el : 0) * S::stride;
  const uint32_t e0 = active ? e : 0;
  const uint32_t node = 8 * (e0 * Np + ijk);
  const BoxElem<D>* rec = box_elem<D>(p, e0);
  for (int t = threadIdx.x; t < NQ * NQ; t += blockDim.x) {
    const int b = t % NQ, a = t / NQ;
    sS[t] = 0.5 * (p.D[b + NQ * a] * p.bw[b] - p.D[a + NQ * b] * p.bw[a]);
  }
  for (int t = threadIdx.x; t < NQ; t += blockDim.x) siw[t] = 1 / p.bw[t];
  int idx[3];
  node_index<D>(ijk, NQ, idx);
  // a node of the upper half of its line in direction r, at line position c >= M, by its position there
  auto half_pos = [&](int r, int c) {
    int pos = 0, st = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      pos += (d == r ? c - M : idx[d]) * st;
      st *= d == r ? M : NQ;
    }
    return pos;
  };
  double q1[Ns], acc[Ns];
  BF bf;
  if (role == D) bf.load(rec, ijk);
  if (role == 0) {
    double a1[NA], P[NPL];
#pragma unroll
    for (int s = 0; s < Ns; ++s) q1[s] = ldo(p, q, s, node);
    box_aux<L>(p, node, a1);
    ep.load(p, node);
    EC::prim(p.c, q1, GRAV ? a1[0] : 0.0, P);
    if (active) {
#pragma unroll
      for (int k = 0; k < NPL; ++k) sP[k * Np + ijk] = P[k];
#pragma unroll
      for (int s = 0; s < Ns; ++s) sP[S::state + s * Np + ijk] = q1[s];
      if constexpr (GRAV) sP[S::state + Ns * Np + ijk] = a1[0];
    }
#pragma unroll
    for (int s = 0; s < Ns; ++s) acc[s] = 0.0;
    if (active) L::sources(p.c, acc, q1, a1, all_dirs<L>(), false);
  }
  __syncthreads();  // tables, primitives and state written
  double vol[Ns];
#pragma unroll
  for (int s = 0; s < Ns; ++s) vol[s] = 0.0;
  const double inv_gm1 = 1 / (p.c.gamma - 1);
#pragma unroll
  for (int m0 = 1; m0 <= M; m0 += BOX_SLOTS) {
    for_dirs<0, D>([&](auto R) {
      constexpr int r = decltype(R)::value, st = line_stride<NQ, r>();
      if (role != r || !active) return;
      const int a = idx[r], lbase = ijk - a * st;
      double P1[NPL];
#pragma unroll
      for (int k = 0; k < NPL; ++k) P1[k] = sP[k * Np + ijk];
#pragma unroll
      for (int m = m0; m < m0 + BOX_SLOTS && m <= M; ++m) {
        const bool hs = HALF && m == M;
        if (hs && a >= M) continue;
        const int b = a + m >= NQ ? a + m - NQ : a + m;
        const int ib = lbase + b * st;
        double P2[NPL], sf[Ns], ta, tb;
#pragma unroll
        for (int k = 0; k < NPL; ++k) P2[k] = sP[k * Np + ib];
        EC::template pair<r>(inv_gm1, P1, P2, sS[b + NQ * a], sf, &ta, &tb);
#pragma unroll
        for (int s = 0; s < Ns; ++s) vol[s] += sf[s];
        if (GRAV) {
          vol[1 + r] -= ta;
          sf[1 + r] += tb;
        }
        // the partner's share, which it subtracts
        double* slot = sP + S::xch + r * S::share + (m - 1) * Ns * Np + (hs ? half_pos(r, b) : ib);
        const int xs = hs ? Np / 2 : Np;
#pragma unroll
        for (int s = 0; s < Ns; ++s) slot[s * xs] = sf[s];
      }
    });
    if (m0 == 1 && role == D && active) bf.run(p, rec, e, ijk, q, sP + S::faces, sP + S::state, siw[0]);
    __syncthreads();  // the round's shares, and the face fluxes, written
    for_dirs<0, D>([&](auto R) {
      constexpr int r = decltype(R)::value;
      if (role != r || !active) return;
      const int a = idx[r];
#pragma unroll
      for (int m = m0; m < m0 + BOX_SLOTS && m <= M; ++m) {
        const bool hs = HALF && m == M;
        if (hs && a < M) continue;
        const double* slot = sP + S::xch + r * S::share + (m - 1) * Ns * Np + (hs ? half_pos(r, a) : ijk);
        const int xs = hs ? Np / 2 : Np;
#pragma unroll
        for (int s = 0; s < Ns; ++s) vol[s] -= slot[s * xs];
      }
    });
  }
  if (active && role > 0 && role < D) {
#pragma unroll
    for (int s = 0; s < Ns; ++s) sP[S::sum + ((role - 1) * Ns + s) * Np + ijk] = vol[s];
  }
  __syncthreads();  // the later directions' sums written
  if (!active || role > 0) return;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const double gw = rec->g[d] * siw[idx[d]];
#pragma unroll
    for (int s = 0; s < Ns; ++s) acc[s] = fma(gw, d == 0 ? vol[s] : sP[S::sum + ((d - 1) * Ns + s) * Np + ijk], acc[s]);
  }
#pragma unroll
  for (int s = 0; s < Ns; ++s) acc[s] = ep.start_fused(s, acc[s]);
  BF::gather(idx, sP + S::faces, acc);
  ep.store(p, node, q1, acc);
}

template <class L, int NQ, int SF>
ATM_DEV void fast_box_body(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q,
                           double* __restrict__ dq, double alpha, int assign, double* __restrict__ qout, double bdt,
                           int epw) {
  StageEnd<L> ep(dq, alpha, assign, qout, bdt);
  fast_box_node<L, NQ, SF>(p, lds, blk, q, ep, epw);
}

template <class L, int NQ, int SF>
struct FastBoxBody {
  template <class EP>
  ATM_DEV static void run(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep, int epw) {
    fast_box_node<L, NQ, SF>(p, lds, blk, q, ep, epw);
  }
};

template <class L, int NQ, int SF>
__global__ void __attribute__((amdgpu_flat_work_group_size(1, fast_max_threads<L, NQ, SF>())))
fast_box_ark_kernel(const DevDG p, const DevDG pl, const double* __restrict__ q, const ArkSums a, int epw) {
  extern __shared__ double lds[];
  box_ark_pair<L, NQ, FastBoxBody<L, NQ, SF>>(p, pl, lds, q, a, epw);
}

template <class L, int NQ, int SF>
hipError_t launch_fast_box_ark(const DevDG& p, const DevDG& pl, hipStream_t st, const double* q, const ArkSums& a) {
  return launch_box_ark_pair<L, NQ>(fast_box_ark_kernel<L, NQ, SF>, fast_max_threads<L, NQ, SF>(), p, pl, st, q, a);
}

template <class L, int NQ, int SF>
__global__ void __attribute__((amdgpu_flat_work_group_size(1, fast_max_threads<L, NQ, SF>())))
fast_box_kernel(const DevDG p, const double* __restrict__ q, double* __restrict__ dq, double alpha, int assign,
                double* __restrict__ qout, double bdt, int epw) {
  extern __shared__ double lds[];
  fast_box_body<L, NQ, SF>(p, lds, xcd_block(), q, dq, alpha, assign, qout, bdt, epw);
}

template <class L, int NQ, int SF>
__global__ void __attribute__((amdgpu_flat_work_group_size(1, fast_max_threads<L, NQ, SF>())))
fast_box_kernel_batch(const BatchEntry* __restrict__ tab, int n, int parity, double alpha, int assign, double b,
                      int epw) {
  extern __shared__ double lds[];
  const int64_t lb = xcd_block();
  const int i = batch_find(tab, n, lb);
  const DevDG p = tab[i].p;
  fast_box_body<L, NQ, SF>(p, lds, lb - tab[i].block_start, tab[i].buf[parity], tab[i].dq, alpha, assign,
                           tab[i].buf[1 - parity], b * tab[i].dt, epw);
}

// One launch per stage for members of N = 3..7 (as fd_fast_multi_kernel_batch)
template <class L, int SF>
__global__ void __launch_bounds__(512)
    fast_box_multi_kernel_batch(const BatchEntry* __restrict__ tab, int n, int parity, double alpha, int assign,
                                double b) {
  extern __shared__ double lds[];
  const int64_t lb = xcd_block();
  const int i = batch_find(tab, n, lb);
  const DevDG p = tab[i].p;
  const int64_t blk = lb - tab[i].block_start;
  const double* qin = tab[i].buf[parity];
  double* qo = tab[i].buf[1 - parity];
  const double bdt = b * tab[i].dt;
  switch (p.Nq) {
    case 4: fast_box_body<L, 4, SF>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 5: fast_box_body<L, 5, SF>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 6: fast_box_body<L, 6, SF>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 7: fast_box_body<L, 7, SF>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 8: fast_box_body<L, 8, SF>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    default: break;
  }
}

template <class L, int SF>
hipError_t launch_fast_box_multi_batch(const BatchEntry* tab, int n, int64_t blocks, int threads, size_t lds, int epw,
                                       hipStream_t st, int parity, double alpha, int assign, double b) {
  (void)epw;  // every member carries its own in the table
  hipLaunchKernelGGL((fast_box_multi_kernel_batch<L, SF>), dim3(blocks), dim3(threads), lds, st, tab, n, parity, alpha,
                     assign, b);
  return hipGetLastError();
}

template <class L, int NQ, int SF>
__global__ void __launch_bounds__(1024)
    fast_box_roles_kernel(const DevDG p, const double* __restrict__ q, double* __restrict__ dq, double alpha,
                          int assign, double* __restrict__ qout, double bdt, int epw) {
  extern __shared__ double lds[];
  StageEnd<L> ep(dq, alpha, assign, qout, bdt);
  fast_box_roles_node<L, NQ, SF>(p, lds, xcd_block(), q, ep, epw);
}

// Whether a mesh's elements are dealt out by role: up to a wave per SIMD of the form with a thread per node and
// two workgroups a CU (six waves a CU in 2-D), which a node's chain of pairs bounds.  Per pass of two LSRK54 steps,
// a thread per node against roles: vortex 8^2 N = 4 67 -> 50 us, 20^2 N = 6 77 -> 57, 36^2 N = 6 79 -> 69,
// 32^2 N = 7 77 -> 67, 45^2 N = 4 60 -> 54, bubble 5^3 N = 4 83 -> 64, 8^3 N = 4 100 -> 77, 8^3 N = 3 76 -> 62,
// 6^3 N = 5 100 -> 78; beyond: vortex 45^2 N = 6 85 -> 87, 70^2 N = 6 127 -> 152, bubble 10^3 N = 3 84 -> 88,
// 10^3 N = 4 113 -> 129, 8^3 N = 5 126 -> 149.
// 3-D elements of N = 1 gain nothing (10^3 63 -> 64), those of N = 6 and 7 have too many threads.
template <class L, int NQ>
constexpr bool fast_box_has_roles() {
  return L::D == 2 || (NQ >= 3 && NQ <= 6);
}
template <class L, int NQ>
bool fast_box_roles(const DevDG& p, int blocks, int threads) {
  constexpr int waves = 256 * (L::D == 2 ? 6 : 4);
  return (L::D == 2 || blocks <= 512) && (int64_t)blocks * threads <= 64 * waves && (L::D + 1) * threads <= 1024 &&
         FastRoles<L, NQ>::lds(p.epw) <= 160 * 1024;
}

template <class L, int NQ, int SF>
hipError_t launch_fast_box(const DevDG& p, hipStream_t st, const double* q, double* dq, double alpha, int assign,
                           double* qout, double bdt) {
  constexpr int Np = ipow(NQ, L::D);
  const int threads = ((p.epw * Np + 63) / 64) * 64;
  if (p.epw < 1 || threads > fast_max_threads<L, NQ, SF>()) return hipErrorInvalidConfiguration;
  const int blocks = (p.K + p.epw - 1) / p.epw;
  if (blocks == 0) return hipSuccess;
  if constexpr (fast_box_has_roles<L, NQ>())
    if (fast_box_roles<L, NQ>(p, blocks, threads)) {
      using S = FastRoles<L, NQ>;
      hipLaunchKernelGGL((fast_box_roles_kernel<L, NQ, SF>), dim3(blocks), dim3((L::D + 1) * threads), S::lds(p.epw),
                         st, p, q, dq, alpha, assign, qout, bdt, p.epw);
      return hipGetLastError();
    }
  hipLaunchKernelGGL((fast_box_kernel<L, NQ, SF>), dim3(blocks), dim3(threads), p.lds, st, p, q, dq, alpha, assign,
                     qout, bdt, p.epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF>
hipError_t launch_fast_box_batch(const BatchEntry* tab, int n, int64_t blocks, int threads, size_t lds, int epw,
                                 hipStream_t st, int parity, double alpha, int assign, double b) {
  hipLaunchKernelGGL((fast_box_kernel_batch<L, NQ, SF>), dim3(blocks), dim3(threads), lds, st, tab, n, parity, alpha,
                     assign, b, epw);
  return hipGetLastError();
}

// Default elements per workgroup: one wave of small elements, one element from 64 nodes on (two for the
// 3-D N = 6 ones, see fast_max_threads).  Against workgroups of 256 threads, per stage: 2-D vortex 45^2
// N = 6 9.6 -> 9.1 us, 16^2 N = 5 9.8 -> 8.8, 64^2 N = 3 6.2 -> 5.9, 128^2 N = 4 15.8 -> 15.6; 3-D bubble
// 40^3 N = 1 29.2 -> 27.1, 27^3 N = 2 28.4 -> 28.1: a barrier waits for fewer waves, and a small mesh
// spreads over more CUs.
template <class L, int NQ, int SF>
constexpr int fast_box_epw() {
  constexpr int Np = ipow(NQ, L::D);
  if (fast_max_threads<L, NQ, SF>() > 512) return 2;
  return Np >= 64 ? 1 : 64 / Np;
}

template <class L, int NQ, int SF>
Resolved fast_box_variant() {
  Resolved r = make_resolved(launch_fast_box<L, NQ, SF>, launch_fast_box_batch<L, NQ, SF>, L::Ns,
                             fast_box_epw<L, NQ, SF>(), sizeof(double) * (NQ * NQ + NQ),
                             sizeof(double) * fast_box_elem_doubles<L, NQ>(), fast_max_threads<L, NQ, SF>());
  if constexpr (NQ >= 4 && NQ <= 8) r.mbfn = launch_fast_box_multi_batch<L, SF>;
  if constexpr (L::LAW == ATM_LAW_EULER_GRAVITY) r.pfn = launch_fast_box_ark<L, NQ, SF>;
  return r;
}

template <class L, int SF>
Resolved fast_box_nq(int Nq) {
  switch (Nq) {
    case 2: return fast_box_variant<L, 2, SF>();
    case 3: return fast_box_variant<L, 3, SF>();
    case 4: return fast_box_variant<L, 4, SF>();
    case 5: return fast_box_variant<L, 5, SF>();
    case 6: return fast_box_variant<L, 6, SF>();
    case 7: return fast_box_variant<L, 7, SF>();
    case 8: return fast_box_variant<L, 8, SF>();
    default: return Resolved{nullptr, 0, 0, nullptr, 1};
  }
}

template <template <int> class LAW, int SF>
Resolved fast_box_dims(int dim, int Nq) {
  if (dim == 2) return fast_box_nq<LAW<2>, SF>(Nq);
  if (dim == 3) return fast_box_nq<LAW<3>, SF>(Nq);
  return Resolved{nullptr, 0, 0, nullptr, 1};
}

}  // namespace atm
