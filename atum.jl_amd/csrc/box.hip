// Box elements: detection from an operator's geometry arrays (box.hpp).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "box.hpp"
#include "handles.hpp"

namespace {

constexpr int CAND = 5;  // Jacobians tried: the quotient of the first entry and its weight, and 2 ulps either side

__device__ double candidate(double x, int c) {
  return __longlong_as_double(__double_as_longlong(x) + (c - CAND / 2));
}

// the candidate to keep: the quotient itself if it fits, else any that does
__device__ int pick(unsigned mask) { return (mask >> (CAND / 2)) & 1u ? CAND / 2 : __ffs(mask) - 1; }

// One workgroup per element: writes its record (rec not null), or sets *bad when its arrays are not those of a box.
// lift: the kernels scale what a face adds by g_r / w_end in place of faceMJ MJI, so the face Jacobians have to be
// J g_r.  wp, wf: products of the weights per node and face point.
// Bound by the latency of an element's loads, so none of them waits for another's comparison (with && in place of &
// every one did): 16 2-D elements of N = 2 18 -> 12 us, 6^3 of N = 3 40 -> 14 us, 16^3 of N = 4 60 -> 32 us.
template <int D>
__global__ void __launch_bounds__(256)
    box_detect_kernel(DevDG p, const double* __restrict__ wp, const double* __restrict__ wf, BoxElem<D>* rec, int lift,
                      int32_t* bad) {
  constexpr unsigned ALL = (1u << CAND) - 1;
  __shared__ unsigned mJ, mF[D];
  __shared__ int ok, nb[2 * D];
  for (int64_t e = blockIdx.x; e < p.K; e += gridDim.x) {
    if (threadIdx.x == 0) {
      mJ = ALL;
      for (int r = 0; r < D; ++r) mF[r] = ALL;
      ok = 1;
    }
    __syncthreads();
    const int64_t node0 = e * p.Np, face0 = e * p.Nfp;
    double g0[D], fJ0[D];
    for (int r = 0; r < D; ++r) {
      g0[r] = p.g[(int64_t)(r + D * r) * p.Ntot + node0];
      fJ0[r] = p.faceMJ[face0 + 2 * r * p.Nfpf];
    }
    const double J0 = p.MJ[node0] / wp[0];
    bool good = (J0 > 1e-300) & (J0 < 1e300);
    unsigned m = ALL;
    for (int t = threadIdx.x; t < p.Np; t += blockDim.x) {
      double g[D * D];
      for (int k = 0; k < D * D; ++k) g[k] = p.g[(int64_t)k * p.Ntot + node0 + t];
      const double mj = p.MJ[node0 + t], mji = p.MJI[node0 + t], w = wp[t];
      for (int c = 0; c < CAND; ++c) m &= w * candidate(J0, c) == mj ? ALL : ~(1u << c);
      good &= 1 / mj == mji;
      for (int a = 0; a < D; ++a)
        for (int c = 0; c < D; ++c) good &= g[a + D * c] == (a == c ? g0[a] : 0.0);
    }
    unsigned mf[D];
    for (int r = 0; r < D; ++r) {
      mf[r] = ALL;
      fJ0[r] /= wf[0];
      good &= (fJ0[r] > 1e-300) & (fJ0[r] < 1e300);
    }
    for (int f = threadIdx.x; f < p.Nfp; f += blockDim.x) {
      const int face = f / p.Nfpf, fp = f - face * p.Nfpf, r = face >> 1, side = face & 1;
      double n[D];
      for (int d = 0; d < D; ++d) n[d] = p.normal[d * p.NF + face0 + f];
      const double fMJ = p.faceMJ[face0 + f], w = wf[fp];
      const int tag = p.bctag[e * (2 * D) + face];
      const int64_t ixp = p.faceix_p[face0 + f], ixp0 = p.faceix_p[face0 + face * p.Nfpf];
      // the same point of the opposite face of one element; pos0: its first
      int st = 1, pos = 0, pos0 = 0, rem = fp;
      for (int d = 0; d < D; ++d) {
        good &= n[d] == (d == r ? (side ? 1.0 : -1.0) : 0.0);
        if (d == r) {
          pos0 = (side ? 0 : p.Nq - 1) * st;
          for (int c = 0; c < CAND; ++c) mf[d] &= w * candidate(fJ0[d], c) == fMJ ? ALL : ~(1u << c);
        } else {
          pos += (rem % p.Nq) * st;
          rem /= p.Nq;
        }
        st *= p.Nq;
      }
      good &= (tag != 0) | (ixp == ixp0 + pos);
      if (fp == 0) {
        const int64_t en = ixp / p.Np;
        good &= (tag != 0) | (ixp == en * p.Np + pos0);
        nb[face] = tag ? -tag : (int)en;
      }
    }
    atomicAnd(&mJ, m);
    for (int r = 0; r < D; ++r) atomicAnd(&mF[r], mf[r]);
    if (!good) ok = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
      bool box = ok && mJ;
      for (int r = 0; r < D; ++r) box = box && mF[r];
      BoxElem<D> x;
      x.J = candidate(J0, pick(mJ));
      for (int r = 0; r < D; ++r) {
        x.g[r] = g0[r];
        x.fJ[r] = candidate(fJ0[r], pick(mF[r]));
        // (a box's own are a few roundings apart)
        if (lift) box = box && fabs(x.g[r] * x.J - x.fJ[r]) <= 64 * 2.220446049250313e-16 * x.fJ[r];
      }
      if (!box) *bad = 1;
      if (box && rec) {
        for (int f = 0; f < 2 * D; ++f) x.nb[f] = nb[f];
        rec[e] = x;
      }
    }
    __syncthreads();
  }
}

template <int D>
hipError_t launch_detect(const DevDG& p, const double* bw, void* rec, int lift, int32_t* bad) {
  hipLaunchKernelGGL(box_detect_kernel<D>, dim3(p.K < 65536 ? p.K : 65536), dim3(p.Np > 128 ? 256 : 64), 0, nullptr, p,
                     bw + p.Nq, bw + p.Nq + p.Np, static_cast<BoxElem<D>*>(rec), lift, bad);
  return hipGetLastError();
}

// LGL weights 2 / (N (N+1) P_N(x)^2), the nodes by Newton on P_N' in extended precision
void lgl_weights(int Nq, double* w) {
  const int N = Nq - 1;
  auto legendre = [](int n, long double x) {
    long double a = 1, b = x;
    if (n == 0) return a;
    for (int k = 2; k <= n; ++k) {
      const long double c = ((2 * k - 1) * x * b - (k - 1) * a) / k;
      a = b;
      b = c;
    }
    return b;
  };
  for (int i = 0; i < Nq; ++i) {
    long double P = 1;
    if (i > 0 && i < N) {
      long double x = -std::cos(3.14159265358979323846L * i / N);
      for (int it = 0; it < 30; ++it) {
        const long double p0 = legendre(N, x), p1 = legendre(N - 1, x);
        const long double dP = N * (p1 - x * p0) / (1 - x * x);
        const long double d2P = (2 * x * dP - N * (N + 1) * p0) / (1 - x * x);
        x -= dP / d2P;
      }
      P = legendre(N, x);
    }
    w[i] = (double)(2 / (N * (N + 1) * P * P));
  }
}

}  // namespace

namespace atm {

std::vector<double> box_tables(int dim, int Nq, const double* w) {
  const int Np = ipow(Nq, dim), Nfpf = Np / Nq;
  std::vector<double> tab((size_t)Nq + Np + Nfpf);
  std::memcpy(tab.data(), w, sizeof(double) * Nq);
  for (int t = 0; t < Np + Nfpf; ++t) {
    int rem = t < Np ? t : t - Np;
    double v = 1.0;
    for (int i = 0; i < (t < Np ? dim : dim - 1); ++i) {
      v = v * w[rem % Nq];
      rem /= Nq;
    }
    tab[(size_t)Nq + t] = v;
  }
  return tab;
}

bool box_kernels(const atm_dg* dg, const atm_dg_desc* d, Resolved* r) {
  if (dg->dev.K < 1 || !box_fits(dg->dim, dg->Np, dg->Ns, dg->dev.K)) return false;
  *r = resolve_box(d, dg->Nq);
  return r->fn && r->lds <= dg->ctx->max_lds;
}

void dg_use_box(atm_dg* dg, const Resolved& r, const void* rec, const double* tab) {
  DevDG& p = dg->dev;
  p.box = rec;
  p.bw = tab;
  dg->fn = r.fn;
  dg->bfn = r.bfn;
  dg->mbfn = r.mbfn;
  dg->afn = r.afn;
  dg->pfn = r.pfn;
  dg->lds = r.lds;
  dg->epw = r.epw;
  dg->lds_fixed = r.lds_fixed;
  dg->lds_elem = r.lds_elem;
  dg->max_threads = r.max_threads;
  p.epw = r.epw;
  p.lds = (int)r.lds;
}

// whether the operator's kernels are FAST ones, which read neither Jacobians nor face Jacobians
static int box_lift(const atm_dg_desc* d) {
  return d->volume_form == ATM_FORM_FLUX_DIFFERENCING && d->precision == ATM_PRECISION_FAST;
}

// Geometry arrays that fit one copy of this size go in one allocation and one copy: each array's own takes 8 us,
// whatever its size.  An operator of 16 2-D elements of N = 2: 184 -> 85 us with the shorter look-over.
constexpr size_t PACKED_UPLOAD = 256 << 10;

int dg_upload_geometry(atm_dg* dg, const atm_dg_desc* d) {
  DevDG& p = dg->dev;
  atm_ctx* ctx = dg->ctx;
  const int dim = dg->dim, Nq = dg->Nq, Np = dg->Np;
  const size_t N = (size_t)p.Ntot, NF = (size_t)p.NF;
  Resolved r;
  const bool look = box_kernels(dg, d, &r);
  // one upload: D and, where there are box kernels, the weight tables and the flag that box_detect_kernel raises
  if (!d->D) return fail(ctx, ATM_ERR_ARG, "missing array");
  std::vector<double> tab(d->D, d->D + Nq * Nq);
  const size_t at_w = tab.size();
  if (look) {
    double w[8];
    lgl_weights(Nq, w);
    const std::vector<double> wt = box_tables(dim, Nq, w);
    tab.insert(tab.end(), wt.begin(), wt.end());
    tab.push_back(0.0);
  }
  const struct {
    const void* host;
    size_t bytes;
  } pieces[] = {{tab.data(), tab.size() * sizeof(double)},
                {d->g, dim * dim * N * sizeof(double)},
                {d->MJ, N * sizeof(double)},
                {d->MJI, N * sizeof(double)},
                {d->faceMJ, NF * sizeof(double)},
                {d->normal, dim * NF * sizeof(double)},
                {d->faceix_p, NF * sizeof(int64_t)},
                {d->bctag, (size_t)2 * dim * p.K * sizeof(int32_t)}};
  const char* dev[8] = {};
  auto padded = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
  size_t total = 0;
  for (const auto& x : pieces) total += padded(x.bytes);
  int rc = ATM_OK;
  if (total <= PACKED_UPLOAD) {
    std::vector<char> host(total);
    size_t at = 0;
    for (const auto& x : pieces) {
      if (x.bytes) std::memcpy(host.data() + at, x.host, x.bytes);
      at += padded(x.bytes);
    }
    const char* base = nullptr;
    if ((rc = upload_copy(dg, host.data(), total, &base))) return rc;
    at = 0;
    for (int i = 0; i < 8; ++i) {
      if (pieces[i].bytes) dev[i] = base + at;
      at += padded(pieces[i].bytes);
    }
  } else {
    for (int i = 0; i < 8; ++i)
      if ((rc = upload_copy(dg, static_cast<const char*>(pieces[i].host), pieces[i].bytes, &dev[i]))) return rc;
  }
  p.D = (const double*)dev[0];
  p.g = (const double*)dev[1];
  p.MJ = (const double*)dev[2];
  p.MJI = (const double*)dev[3];
  p.faceMJ = (const double*)dev[4];
  p.normal = (const double*)dev[5];
  p.faceix_p = (const int64_t*)dev[6];
  p.bctag = (const int32_t*)dev[7];
  if (!look) return ATM_OK;
  // On the null stream, as the uploads: creating an operator waits for nothing that is queued on the context's
  // stream.  The records are allocated once every element is a box (freeing them again would wait for the device).
  const double* bw = p.D + at_w;
  int32_t* bad = reinterpret_cast<int32_t*>(const_cast<double*>(p.D) + tab.size() - 1);
  const int lift = box_lift(d);
  auto detect = [&](void* rec) {
    if (dim == 1) return launch_detect<1>(p, bw, rec, lift, bad);
    if (dim == 2) return launch_detect<2>(p, bw, rec, lift, bad);
    return launch_detect<3>(p, bw, rec, lift, bad);
  };
  int32_t host_bad = 1;
  HIPCHK(ctx, detect(nullptr));
  HIPCHK(ctx, hipMemcpy(&host_bad, bad, sizeof(int32_t), hipMemcpyDeviceToHost));
  if (host_bad) return ATM_OK;
  void* rec = nullptr;
  if ((rc = dg_alloc(dg, box_elem_bytes(dim) * (size_t)p.K, &rec))) return rc;
  HIPCHK(ctx, detect(rec));
  HIPCHK(ctx, hipStreamSynchronize(nullptr));
  dg_use_box(dg, r, rec, bw);
  return ATM_OK;
}

Resolved resolve_box_weak_euler(int dim, int mask, int Nq);
Resolved resolve_box_weak_euler_gravity(int dim, int mask, int Nq);
Resolved resolve_box_weak_linear(int dim, int mask, int Nq);
Resolved resolve_box_weak_shallow_water(int dim, int mask, int Nq);

#define ATM_BOX_EC(FORM, LAW) \
  Resolved resolve_box_##FORM##_##LAW##_roe(int dim, int Nq); \
  Resolved resolve_box_##FORM##_##LAW##_rusanov(int dim, int Nq);
ATM_BOX_EC(fast, euler)
ATM_BOX_EC(fast, euler_gravity)
ATM_BOX_EC(fd, euler)
ATM_BOX_EC(fd, euler_gravity)

// Kernels for an operator whose elements are all boxes (fn == nullptr: the general ones)
Resolved resolve_box(const atm_dg_desc* d, int Nq) {
  if (d->volume_form == ATM_FORM_WEAK && d->surface_flux == ATM_FLUX_RUSANOV) switch (d->law) {
      case ATM_LAW_ADVECTION: return weak_box_dims<Advection, ATM_FLUX_RUSANOV, true>(d->dim, d->dirmask, Nq);
      case ATM_LAW_EULER: return resolve_box_weak_euler(d->dim, d->dirmask, Nq);
      case ATM_LAW_EULER_GRAVITY: return resolve_box_weak_euler_gravity(d->dim, d->dirmask, Nq);
      case ATM_LAW_LINEAR_EULER_GRAVITY: return resolve_box_weak_linear(d->dim, d->dirmask, Nq);
      case ATM_LAW_SHALLOW_WATER: return resolve_box_weak_shallow_water(d->dim, d->dirmask, Nq);
      default: break;
    }
  if (d->volume_form == ATM_FORM_FLUX_DIFFERENCING && d->volume_flux == ATM_FLUX_EC &&
      d->fd_kernel == ATM_FD_PER_DIR && d->dirmask == (1 << d->dim) - 1 &&
      (d->surface_flux == ATM_FLUX_ROE || d->surface_flux == ATM_FLUX_RUSANOV)) {
    const bool roe = d->surface_flux == ATM_FLUX_ROE, grav = d->law == ATM_LAW_EULER_GRAVITY;
    if (!grav && d->law != ATM_LAW_EULER) return Resolved{nullptr, 0, 0, nullptr, 1};
    if (d->precision == ATM_PRECISION_FAST && d->dim >= 2) {  // FAST precision has no 1-D kernels of its own
      if (grav) return roe ? resolve_box_fast_euler_gravity_roe(d->dim, Nq) : resolve_box_fast_euler_gravity_rusanov(d->dim, Nq);
      return roe ? resolve_box_fast_euler_roe(d->dim, Nq) : resolve_box_fast_euler_rusanov(d->dim, Nq);
    }
    if (grav) return roe ? resolve_box_fd_euler_gravity_roe(d->dim, Nq) : resolve_box_fd_euler_gravity_rusanov(d->dim, Nq);
    return roe ? resolve_box_fd_euler_roe(d->dim, Nq) : resolve_box_fd_euler_rusanov(d->dim, Nq);
  }
  return Resolved{nullptr, 0, 0, nullptr, 1};
}

}  // namespace atm

extern "C" int atm_box_elements_fit(int dim, int N, int Ns, int64_t K) {
  if (dim < 1 || dim > 3 || N < 1 || N > 7 || Ns < 1 || K < 0) return ATM_ERR_ARG;
  return atm::box_fits(dim, atm::ipow(N + 1, dim), Ns, K) ? 1 : 0;
}

extern "C" int atm_dg_box_elements(const atm_dg* dg) { return !dg ? ATM_ERR_ARG : dg->dev.box ? 1 : 0; }
