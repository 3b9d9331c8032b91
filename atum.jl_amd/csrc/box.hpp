// Box elements: the compact geometry of axis-aligned rectangular elements.
//
// Every element of a brick mesh is an axis-aligned box: its metric is the diagonal 2/h in
// every node, MJ and faceMJ are the element's Jacobians times products of the LGL weights,
// its normals are the unit vectors and a face's neighbour nodes are the opposite face of one
// element in the same order.  The element kernels of such an operator read one BoxElem per
// element instead of d^2 + 2 doubles per node and d + 2 per face point: for 2-D N = 3 that is
// 56 bytes per element of 16 nodes instead of 1280 (the state, dq and the new state are 2048).
//
// Whether an operator's elements are boxes is found from its geometry arrays when it is
// created (box_detect_kernel): the values that the compact form reproduces have to equal the arrays
// bit for bit in every node and face point, so that both forms of a kernel compute with the
// same numbers; for the FAST kernels, which use 2/h for faceMJ MJI too (box_fast.hpp), the face
// Jacobians also have to be the Jacobian times 2/h.  Operators with any other element keep the
// general kernels.
#pragma once
#include <algorithm>
#include <type_traits>

#include "dg_kernels.hpp"
#include "fast_flux.hpp"

namespace atm {

template <int D>
struct BoxElem {
  double g[D];        // 2/h: the diagonal of the metric
  double J;           // MJ = wp * J, wp the product of the node's LGL weights; MJI = 1/MJ
  double fJ[D];       // faceMJ = wf * fJ[r] on the faces of direction r
  int32_t nb[2 * D];  // neighbour element of each face, or minus the boundary tag
};

// The box kernels address fields and records with 32-bit byte offsets from a uniform base (a scalar register and
// one vector register per address instead of 64-bit vector arithmetic for every load), so they take operators
// whose state is below 4 GB and whose records end there (one component at N = 1, in 1-D also N = 2, has larger
// records than states); larger ones run the general kernels.  Np: nodes of an element, Ns: components.
constexpr int64_t BOX_MAX_STATE = (int64_t)1 << 29;    // doubles
constexpr int64_t BOX_MAX_RECORDS = (int64_t)1 << 32;  // bytes
constexpr size_t box_elem_bytes(int dim) {
  return (size_t)(2 * dim + 1) * sizeof(double) + (size_t)2 * dim * sizeof(int32_t);
}
static_assert(sizeof(BoxElem<1>) == box_elem_bytes(1) && sizeof(BoxElem<2>) == box_elem_bytes(2) &&
              sizeof(BoxElem<3>) == box_elem_bytes(3));
constexpr bool box_fits(int dim, int64_t Np, int64_t Ns, int64_t K) {
  return K < BOX_MAX_STATE && Ns * Np * K < BOX_MAX_STATE && K * (int64_t)box_elem_bytes(dim) <= BOX_MAX_RECORDS;
}

// A global pointer kept in scalar registers: the empty statement hides it from the address arithmetic
// of the lanes, so that a load takes it as the base and the lane's offset as one register.
typedef const char __attribute__((address_space(1))) * gptr;
ATM_DEV gptr uniform(const void* b) {
  gptr g = (gptr)b;
  asm("" : "+s"(g));
  return g;
}
ATM_DEV double ldg(gptr b, uint32_t off) { return *(const double __attribute__((address_space(1)))*)(b + off); }
ATM_DEV void stg(gptr b, uint32_t off, double v) { *(double __attribute__((address_space(1)))*)(char __attribute__((address_space(1)))*)(b + off) = v; }

// component s of a field at a byte offset
ATM_DEV double ldo(const DevDG& p, const double* field, int s, uint32_t off) {
  return ldg(uniform(field + s * p.Ntot), off);
}
ATM_DEV void sto(const DevDG& p, double* field, int s, uint32_t off, double v) {
  stg(uniform(field + s * p.Ntot), off, v);
}

template <int D>
ATM_DEV const BoxElem<D>* box_elem(const DevDG& p, uint32_t e) {
  return reinterpret_cast<const BoxElem<D>*>(static_cast<const char*>(p.box) + e * (uint32_t)sizeof(BoxElem<D>));
}

// load_aux and epilogue with a byte offset of the node
template <class L>
ATM_DEV void box_aux(const DevDG& p, uint32_t off, double* a) {
#pragma unroll
  for (int s = 0; s < L::NA; ++s) a[s] = (s < p.naux) ? ldo(p, p.aux, s, off) : 0.0;
}

template <class L>
ATM_DEV void box_epilogue(const DevDG& p, uint32_t off, const double* q1, const double* acc, double* __restrict__ dq,
                          double* __restrict__ qout, double bdt) {
#pragma unroll
  for (int s = 0; s < L::Ns; ++s) {
    sto(p, dq, s, off, acc[s]);
    if (qout) sto(p, qout, s, off, q1[s] + bdt * acc[s]);
  }
}

__host__ __device__ constexpr int ipow(int b, int n) { return n == 0 ? 1 : b * ipow(b, n - 1); }

// The direction mask of an operator of all directions
template <class L>
constexpr int all_dirs() {
  return (1 << L::D) - 1;
}

// Line stride of direction R in an element's node numbering
template <int NQ, int R>
constexpr int line_stride() {
  return ipow(NQ, R);
}

// Compile-time loop over the directions
template <int R, int D, class F>
ATM_DEV void for_dirs(F&& f) {
  if constexpr (R < D) {
    f(std::integral_constant<int, R>{});
    for_dirs<R + 1, D>(f);
  }
}

// What the weak form takes of a state: row<R>() is the law's flux in direction R, speed<R>() its wave speed with
// the unit normal of direction R.  A node forms its own once, for its flux and all its faces.  The quotients by
// one density share a reciprocal and are corrected (fast_div), so they and the roots (fast_sqrt) are the law's.
template <class L, int LAW = L::LAW>
struct WeakSide;

template <class L>
struct WeakSide<L, ATM_LAW_ADVECTION> {
  ATM_DEV WeakSide(const LawConst&, const double*, const double*) {}
  template <int R>
  ATM_DEV void row(const LawConst& c, const double* q, double* f) const { f[0] = c.u[R] * q[0]; }
  template <int R>
  ATM_DEV double speed(const LawConst& c) const { return fabs(c.u[R]); }
};

// root of a squared sound speed: fast_sqrt, and 0 for 0
ATM_DEV double speed_root(double x) { return x == 0 ? x : fast_sqrt(x); }

template <class L>
struct WeakSide<L, ATM_LAW_LINEAR_EULER_GRAVITY> {
  static constexpr int D = L::D;
  double p, h, cs;
  ATM_DEV WeakSide(const LawConst& c, const double* q, const double* a) {
    const double phi = a[0], rho = a[D + 1], ref_p = a[D + 2], gm1 = c.gamma - 1;
    const double ir = rcp_div(rho);
    p = gm1 * (q[D + 1] - q[0] * phi);
    const double ref_rhoe = fast_div(ref_p, gm1, rcp_div(gm1)) + rho * phi;
    h = fast_div(ref_rhoe + ref_p, rho, ir);
    cs = speed_root(fast_div(c.gamma * ref_p, rho, ir));
  }
  template <int R>
  ATM_DEV void row(const LawConst&, const double* q, double* f) const {
    f[0] = q[1 + R];
#pragma unroll
    for (int d = 0; d < D; ++d) f[1 + d] = d == R ? p : 0.0;
    f[D + 1] = h * q[1 + R];
  }
  template <int R>
  ATM_DEV double speed(const LawConst&) const { return cs; }
};

// the laws with velocities: Euler, with or without gravity, and shallow water
template <class L, int LAW>
struct WeakSide {
  static constexpr int D = L::D;
  static constexpr bool SW = LAW == ATM_LAW_SHALLOW_WATER, GRAV = LAW == ATM_LAW_EULER_GRAVITY;
  double u[D], p, dp, cs;  // velocity, pressure, pressure in the momentum flux, sound speed
  ATM_DEV WeakSide(const LawConst& c, const double* q, const double* a) {
    const double rho = q[0], ir = rcp_div(rho);
#pragma unroll
    for (int d = 0; d < D; ++d) u[d] = fast_div(q[1 + d], rho, ir);
    if constexpr (SW) {
      p = dp = c.grav * (rho * rho) / 2;
      cs = speed_root(c.grav * rho);
    } else {
      const double k = 0.5 * fast_div(dotv<D>(q + 1, q + 1), rho, ir);
      p = GRAV ? (c.gamma - 1) * (q[D + 1] - k - rho * a[0]) : (c.gamma - 1) * (q[D + 1] - k);
      dp = p;
      if constexpr (GRAV)
        if (c.pde_level_balance) dp -= a[D + 2];
      cs = speed_root(fast_div(c.gamma * p, rho, ir));
    }
  }
  template <int R>
  ATM_DEV void row(const LawConst&, const double* q, double* f) const {
    f[0] = q[1 + R];
#pragma unroll
    for (int d = 0; d < D; ++d) f[1 + d] = d == R ? q[1 + R] * u[d] + dp : q[1 + R] * u[d];
    f[D + 1] = SW ? u[R] * q[D + 1] : u[R] * (q[D + 1] + p);
  }
  template <int R>
  ATM_DEV double speed(const LawConst&) const { return fabs(u[R]) + cs; }
};

// Surface contributions of the faces this node lies on, subtracted from acc (surface_node on
// box elements).  sw: the LGL weights.
template <class L, int NQ, int MASK>
ATM_DEV void box_surface_node(const DevDG& p, const BoxElem<L::D>& b, uint32_t e, int ijk, const int idx[3],
                              const double* q, const double* qn, const double* an, const WeakSide<L>& own, double MJIn,
                              const double* sw, double* acc) {
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA, Np = ipow(NQ, D);
  for_dirs<0, D>([&](auto R) {
    constexpr int r = decltype(R)::value;
    if constexpr (((MASK >> r) & 1) == 0) return;
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
      boundarystate<L>(p.c, n, qn, -nb, qp);
#pragma unroll
      for (int s = 0; s < NA; ++s) ap[s] = an[s];
    }
    // Rusanov with the normal sg * e_r: the products with the normal's zeros and ones are left out, so the
    // result is the same value (up to the sign of a zero)
    const WeakSide<L> other(p.c, qp, ap);
    double fn[Ns], fp[Ns];
    own.template row<r>(p.c, qn, fn);
    other.template row<r>(p.c, qp, fp);
    const double ws = fmax(own.template speed<r>(p.c), other.template speed<r>(p.c));
#pragma unroll
    for (int s = 0; s < Ns; ++s) nf[s] = sg * ((fn[s] + fp[s]) / 2) - ws * (qp[s] - qn[s]) / 2;
    double wf = 1.0;
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d != r) wf = wf * sw[idx[d]];
    const double fMJ = wf * b.fJ[r];
#pragma unroll
    for (int s = 0; s < Ns; ++s) acc[s] -= fMJ * nf[s] * MJIn;
  });
}

// ---------------------------------------------------------------------------
// Weak form on box elements: weak_body with the compact geometry, the same operations in the
// same order.  Only the flux row of a direction enters its sum (the metric is diagonal), and
// LDS holds only the directions of the operator (the bits of MASK, fixed at compile time).
// Bound by vector instructions and memory traffic about equally (3-D Euler, N = 4: 830 instructions a
// wave, the vector units 70 % busy; they were 1195 when every face formed both sides' law terms with IEEE
// divisions).  Against the general kernels, per fused stage: 2-D shallow water, 256^2 elements, N = 3:
// 42.1 -> 25.9 us (134 MB of states: 5.2 TB/s); 3-D Euler, 20^3, N = 4, which had run the runtime-degree
// kernel: 93.0 -> 39.5 us; 2-D advection, 80^2, N = 4: 6.6 -> 4.6 us.
// The sum over n stays a loop: unrolled, its LDS reads in flight took 30 registers more, which cost
// waves: 40 shallow-water meshes of mixed degree 920 -> 846 us, 3-D Euler 9^3, N = 7 248 -> 195 us a pass
// of 10 stages, shallow water 175^2, N = 7 500 -> 479 us; no size measured was slower by more than 2 %.
// EP: what a node's tendency goes into; load() is called with the node's other loads, store() last.
template <class L, int NQ, int SF, int MASK, class EP>
ATM_DEV void weak_box_node(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q, EP& ep, int epw) {
  static_assert(SF == ATM_FLUX_RUSANOV, "box_surface_node is Rusanov's");
  constexpr int D = L::D, Ns = L::Ns, NA = L::NA, Np = ipow(NQ, D);
  double* sD = lds;
  double* sw = lds + NQ * NQ;
  constexpr int dirs = __builtin_popcount(MASK);
  const int tid = threadIdx.x;
  const int el = tid / Np;
  const int ijk = tid - el * Np;
  const uint32_t le = (uint32_t)blk * epw + el;  // position in the processing order
  const bool active = el < epw && le < (uint32_t)p.K;
  const uint32_t e = (p.sched && active) ? (uint32_t)p.sched[le] : le;
  double* slF = lds + NQ * NQ + NQ + el * (dirs * Ns * Np);  // [dir slot][s][node]
  for (int t = tid; t < NQ * NQ; t += blockDim.x) sD[t] = p.D[t];
  for (int t = tid; t < NQ; t += blockDim.x) sw[t] = p.bw[t];
  double q1[Ns], a1[NA];
  const uint32_t el_e = active ? e : 0;  // a lane past the last element reads element 0 and discards it
  const uint32_t node = 8 * (el_e * Np + ijk);
  int idx[3];
  node_index<D>(ijk, NQ, idx);
  // every load first and unconditionally: the element's record, state, aux and the stage's dq in flight together
  const BoxElem<D> b = *box_elem<D>(p, el_e);
#pragma unroll
  for (int s = 0; s < Ns; ++s) q1[s] = ldo(p, q, s, node);
  box_aux<L>(p, node, a1);
  const double wp = p.bw[NQ + ijk];
  ep.load(p, node);
  const double MJn = wp * b.J;
  const WeakSide<L> own(p.c, q1, a1);
  if (active) {
    for_dirs<0, D>([&](auto R) {
      constexpr int r = decltype(R)::value, slot = __builtin_popcount(MASK & ((1 << r) - 1));
      if constexpr ((MASK >> r) & 1) {
        double F[Ns];
        own.template row<r>(p.c, q1, F);
#pragma unroll
        for (int s = 0; s < Ns; ++s) slF[(slot * Ns + s) * Np + ijk] = b.g[r] * F[s] * MJn;
      }
    });
  }
  __syncthreads();
  if (!active) return;
  const double MJIn = fast_div(1.0, MJn, rcp_div(MJn));
  double dl[Ns];
#pragma unroll
  for (int s = 0; s < Ns; ++s) dl[s] = -0.0;
  L::sources(p.c, dl, q1, a1, MASK, true);
#pragma unroll 1
  for (int n = 0; n < NQ; ++n) {
    double Dn[D];
#pragma unroll
    for (int r = 0; r < D; ++r) Dn[r] = sD[n + NQ * idx[r]] * MJIn;
#pragma unroll
    for (int s = 0; s < Ns; ++s) {
      int slot = 0;
      int st = 1;
#pragma unroll
      for (int r = 0; r < D; ++r) {
        if ((MASK >> r) & 1) {
          dl[s] += Dn[r] * slF[(slot * Ns + s) * Np + ijk + (n - idx[r]) * st];
          ++slot;
        }
        st *= NQ;
      }
    }
  }
  double acc[Ns];
#pragma unroll
  for (int s = 0; s < Ns; ++s) acc[s] = ep.start(s, dl[s]);
  box_surface_node<L, NQ, MASK>(p, b, e, ijk, idx, q, q1, a1, own, MJIn, sw, acc);
  ep.store(p, node, q1, acc);
}

// dq = (assign ? 0 : alpha dq) + L(q) and, with qout, the stage's new state
template <class L>
struct StageEnd {
  double* dq;
  double alpha;
  int assign;
  double* qout;
  double bdt;
  double dq0[L::Ns];
  ATM_DEV StageEnd(double* dq, double alpha, int assign, double* qout, double bdt)
      : dq(dq), alpha(alpha), assign(assign), qout(qout), bdt(bdt) {}
  ATM_DEV void load(const DevDG& p, uint32_t node) {
#pragma unroll
    for (int s = 0; s < L::Ns; ++s) dq0[s] = 0.0;
    if (!assign) {  // uniform over the launch
#pragma unroll
      for (int s = 0; s < L::Ns; ++s) dq0[s] = ldo(p, dq, s, node);
    }
  }
  ATM_DEV double start(int s, double dl) const { return assign ? dl : alpha * dq0[s] + dl; }
  ATM_DEV double start_fused(int s, double dl) const { return assign ? dl : fma(alpha, dq0[s], dl); }
  ATM_DEV void store(const DevDG& p, uint32_t node, const double* q1, const double* acc) const {
    box_epilogue<L>(p, node, q1, acc, dq, qout, bdt);
  }
};

template <class L, int NQ, int SF, int MASK>
ATM_DEV void weak_box_body(const DevDG& p, double* lds, int64_t blk, const double* __restrict__ q,
                           double* __restrict__ dq, double alpha, int assign, double* __restrict__ qout, double bdt,
                           int epw) {
  StageEnd<L> ep(dq, alpha, assign, qout, bdt);
  weak_box_node<L, NQ, SF, MASK>(p, lds, blk, q, ep, epw);
}

// The implicit tendency of an ARK stage, added where it is formed to the sums that the explicit and implicit
// tendencies of the stage go into (ArkSums) instead of being stored and read again by a pass for each
// sum; the same operations in the same order as those passes.
template <class L>
struct ArkEnd {
  const ArkSums& a;
  double ex[L::Ns], in[3][L::Ns];
  ATM_DEV explicit ArkEnd(const ArkSums& a) : a(a) {}
  ATM_DEV void load(const DevDG& p, uint32_t node) {
#pragma unroll
    for (int s = 0; s < L::Ns; ++s) ex[s] = a.ex ? ldo(p, a.ex, s, node) : 0.0;
    load_sums(p, node);
  }
  ATM_DEV void load_sums(const DevDG& p, uint32_t node) {
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (j < a.n && a.in[j]) {
#pragma unroll
        for (int s = 0; s < L::Ns; ++s) in[j][s] = ldo(p, a.in[j], s, node);
      }
  }
  ATM_DEV double start(int, double dl) const { return dl; }
  ATM_DEV void store(const DevDG& p, uint32_t node, const double* q1, const double* im) const {
#pragma unroll
    for (int s = 0; s < L::Ns; ++s) {
      const double e = a.unsplit ? ex[s] - im[s] : ex[s];
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (j < a.n) {
          const double v = a.in[j] ? in[j][s] : q1[s];
          sto(p, a.out[j], s, node, v + a.dt * (a.ea[j] * e + a.ia[j] * im[s]));
        }
    }
  }
};

// An explicit tendency that stays with its node's thread (out: registers)
template <class L>
struct KeepEnd {
  double* out;
  ATM_DEV void load(const DevDG&, uint32_t) {}
  ATM_DEV double start(int, double dl) const { return dl; }
  ATM_DEV double start_fused(int, double dl) const { return dl; }
  ATM_DEV void store(const DevDG&, uint32_t, const double*, const double* acc) const {
#pragma unroll
    for (int s = 0; s < L::Ns; ++s) out[s] = acc[s];
  }
};

// ArkEnd with the explicit tendency given
template <class L>
struct ArkKeptEnd : ArkEnd<L> {
  ATM_DEV ArkKeptEnd(const ArkSums& a, const double* kept) : ArkEnd<L>(a) {
#pragma unroll
    for (int s = 0; s < L::Ns; ++s) this->ex[s] = kept[s];
  }
  ATM_DEV void load(const DevDG& p, uint32_t node) { this->load_sums(p, node); }
};

// The explicit and the implicit tendency of an ARK stage in one launch, for an Euler law with gravity and its
// linearized law in the vertical on the same elements: BODY forms the explicit tendency (an element kernel's
// body, all threads come back from it), which its node's thread keeps, and the weak vertical form follows,
// its state still in the caches.  The same numbers as from two launches, which write and read the
// explicit tendency and read the state again: 32x32x10 elements, N = 3, 29 + 26 us -> 46 us a stage (FAST).
template <class L>
using LinearOf = LinearEulerGravity<L::D>;

template <class L, int NQ, class BODY>
ATM_DEV void box_ark_pair(const DevDG& p, const DevDG& pl, double* lds, const double* __restrict__ q, const ArkSums& a,
                          int epw) {
  using LL = LinearOf<L>;
  const int64_t blk = xcd_block();
  double ex[L::Ns];
#pragma unroll
  for (int s = 0; s < L::Ns; ++s) ex[s] = 0.0;
  KeepEnd<L> keep{ex};
  BODY::run(p, lds, blk, q, keep, epw);
  __syncthreads();  // the explicit form's LDS is free
  ArkKeptEnd<LL> ep(a, ex);
  weak_box_node<LL, NQ, ATM_FLUX_RUSANOV, 1 << (L::D - 1)>(pl, lds, blk, q, ep, epw);
}

template <class L, int NQ, class KERNEL>
hipError_t launch_box_ark_pair(KERNEL kernel, int max_threads, const DevDG& p, const DevDG& pl, hipStream_t st,
                               const double* q, const ArkSums& a) {
  constexpr int Np = ipow(NQ, L::D);
  const int threads = ((p.epw * Np + 63) / 64) * 64;
  if (p.epw < 1 || threads > max_threads) return hipErrorInvalidConfiguration;
  const int blocks = (p.K + p.epw - 1) / p.epw;
  if (blocks == 0) return hipSuccess;
  // the explicit form's LDS holds the implicit one's: the tables and Ns planes of an element
  const int lds = std::max<int>(p.lds, (int)sizeof(double) * (NQ * NQ + NQ + p.epw * L::Ns * Np));
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(threads), lds, st, p, pl, q, a, p.epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF, int MASK>
__global__ void __launch_bounds__(512)
    weak_box_ark_kernel(const DevDG p, const double* __restrict__ q, const ArkSums a, int epw) {
  extern __shared__ double lds[];
  ArkEnd<L> ep(a);
  weak_box_node<L, NQ, SF, MASK>(p, lds, xcd_block(), q, ep, epw);
}

template <class L, int NQ, int SF, int MASK>
hipError_t launch_weak_box_ark(const DevDG& p, hipStream_t st, const double* q, const ArkSums& a) {
  const int threads = ((p.epw * p.Np + 63) / 64) * 64;
  if (p.epw < 1 || threads > 512) return hipErrorInvalidConfiguration;
  const int blocks = (p.K + p.epw - 1) / p.epw;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((weak_box_ark_kernel<L, NQ, SF, MASK>), dim3(blocks), dim3(threads), p.lds, st, p, q, a, p.epw);
  return hipGetLastError();
}

ATM_KERNEL_PAIR(weak_box_kernel, weak_box_body, class L ATM_COMMA int NQ ATM_COMMA int SF ATM_COMMA int MASK,
                L ATM_COMMA NQ ATM_COMMA SF ATM_COMMA MASK)

// One launch per stage for members of different degrees (as weak_multi_kernel_batch)
template <class L, int SF>
__global__ void __launch_bounds__(512)
    weak_box_multi_kernel_batch(const BatchEntry* __restrict__ tab, int n, int parity, double alpha, int assign,
                                double b) {
  extern __shared__ double lds[];
  constexpr int M = all_dirs<L>();
  const int64_t lb = xcd_block();
  const int i = batch_find(tab, n, lb);
  const DevDG p = tab[i].p;
  const int64_t blk = lb - tab[i].block_start;
  const double* qin = tab[i].buf[parity];
  double* qo = tab[i].buf[1 - parity];
  const double bdt = b * tab[i].dt;
  switch (p.Nq) {
    case 4: weak_box_body<L, 4, SF, M>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 5: weak_box_body<L, 5, SF, M>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 6: weak_box_body<L, 6, SF, M>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 7: weak_box_body<L, 7, SF, M>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    case 8: weak_box_body<L, 8, SF, M>(p, lds, blk, qin, tab[i].dq, alpha, assign, qo, bdt, p.epw); break;
    default: break;
  }
}

template <class L, int SF>
hipError_t launch_weak_box_multi_batch(const BatchEntry* tab, int n, int64_t blocks, int threads, size_t lds, int epw,
                                       hipStream_t st, int parity, double alpha, int assign, double b) {
  (void)epw;  // every member carries its own in the table
  hipLaunchKernelGGL((weak_box_multi_kernel_batch<L, SF>), dim3(blocks), dim3(threads), lds, st, tab, n, parity,
                     alpha, assign, b);
  return hipGetLastError();
}

template <class L, int NQ, int SF, int MASK>
hipError_t launch_weak_box(const DevDG& p, hipStream_t st, const double* q, double* dq, double alpha, int assign,
                           double* qout, double bdt) {
  const int threads = ((p.epw * p.Np + 63) / 64) * 64;
  if (p.epw < 1 || threads > 512) return hipErrorInvalidConfiguration;
  const int blocks = (p.K + p.epw - 1) / p.epw;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((weak_box_kernel<L, NQ, SF, MASK>), dim3(blocks), dim3(threads), p.lds, st, p, q, dq, alpha, assign,
                     qout, bdt, p.epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF, int MASK>
hipError_t launch_weak_box_batch(const BatchEntry* tab, int n, int64_t blocks, int threads, size_t lds, int epw,
                                 hipStream_t st, int parity, double alpha, int assign, double b) {
  hipLaunchKernelGGL((weak_box_kernel_batch<L, NQ, SF, MASK>), dim3(blocks), dim3(threads), lds, st, tab, n, parity, alpha,
                     assign, b, epw);
  return hipGetLastError();
}

template <class L, int NQ, int SF, int MASK>
Resolved make_weak_box() {
  constexpr int Np = ipow(NQ, L::D);
  Resolved r = make_resolved(launch_weak_box<L, NQ, SF, MASK>, launch_weak_box_batch<L, NQ, SF, MASK>, L::Ns,
                             elements_per_workgroup(Np), sizeof(double) * (NQ * NQ + NQ),
                             sizeof(double) * __builtin_popcount(MASK) * L::Ns * Np);
  // operators of the last direction only are the implicit halves of IMEX pairs
  if constexpr (L::D > 1 && MASK == 1 << (L::D - 1)) r.afn = launch_weak_box_ark<L, NQ, SF, MASK>;
  return r;
}

template <class L, int SF, int MASK>
Resolved weak_box_nq(int Nq) {
  switch (Nq) {
    case 2: return make_weak_box<L, 2, SF, MASK>();
    case 3: return make_weak_box<L, 3, SF, MASK>();
    case 4: return make_weak_box<L, 4, SF, MASK>();
    case 5: return make_weak_box<L, 5, SF, MASK>();
    case 6: return make_weak_box<L, 6, SF, MASK>();
    case 7: return make_weak_box<L, 7, SF, MASK>();
    case 8: return make_weak_box<L, 8, SF, MASK>();
    default: return Resolved{nullptr, 0, 0, nullptr, 1};
  }
}

// VERT: with the kernels of operators of the last direction only (the implicit half of an IMEX
// pair) beside those of all directions; any other subset runs the general kernels
template <class L, int SF, bool VERT>
Resolved weak_box_mask(int mask, int Nq) {
  if (mask == all_dirs<L>()) return weak_box_nq<L, SF, all_dirs<L>()>(Nq);
  if constexpr (VERT && L::D > 1)
    if (mask == 1 << (L::D - 1)) return weak_box_nq<L, SF, 1 << (L::D - 1)>(Nq);
  return Resolved{nullptr, 0, 0, nullptr, 1};
}

template <template <int> class LAW, int SF, bool VERT>
Resolved weak_box_dims(int dim, int mask, int Nq) {
  if (dim == 1) return weak_box_mask<LAW<1>, SF, VERT>(mask, Nq);
  if (dim == 2) return weak_box_mask<LAW<2>, SF, VERT>(mask, Nq);
  return weak_box_mask<LAW<3>, SF, VERT>(mask, Nq);
}

}  // namespace atm
