// Box elements: detection from an operator's geometry arrays (box.hpp).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "box.hpp"
#include "handles.hpp"

namespace {

// The record of direction count `dim` at `rec`, written field by field (BoxElem<dim>'s layout)
__device__ void store_record(char* rec, int dim, const double* g, double J, const double* fJ, const int32_t* nb) {
  double* d = reinterpret_cast<double*>(rec);
  for (int r = 0; r < dim; ++r) d[r] = g[r];
  d[dim] = J;
  for (int r = 0; r < dim; ++r) d[dim + 1 + r] = fJ[r];
  int32_t* n = reinterpret_cast<int32_t*>(d + 2 * dim + 1);
  for (int f = 0; f < 2 * dim; ++f) n[f] = nb[f];
}

constexpr int CAND = 5;  // Jacobians tried: the quotient of the first entry and its weight, and 2 ulps either side

__device__ double candidate(double x, int c) {
  return __longlong_as_double(__double_as_longlong(x) + (c - CAND / 2));
}

// the candidate to keep: the quotient itself if it fits, else any that does
__device__ int pick(unsigned mask) { return (mask >> (CAND / 2)) & 1u ? CAND / 2 : __ffs(mask) - 1; }

// One workgroup per element: writes its record, or sets *bad when its arrays are not those of a box.  lift: the
// kernels scale what a face adds by g_r / w_end in place of faceMJ MJI, so the face Jacobians have to be J g_r.
__global__ void __launch_bounds__(256)
    box_detect_kernel(DevDG p, int dim, const double* __restrict__ wp, const double* __restrict__ wf, char* rec,
                      int bytes, int lift, int32_t* bad) {
  __shared__ unsigned mJ, mF[3];
  __shared__ int ok;
  for (int64_t e = blockIdx.x; e < p.K; e += gridDim.x) {
    if (threadIdx.x == 0) {
      mJ = mF[0] = mF[1] = mF[2] = (1u << CAND) - 1;
      ok = 1;
    }
    __syncthreads();
    bool good = true;
    const double J0 = p.MJ[e * p.Np] / wp[0];
    good = good && J0 > 1e-300 && J0 < 1e300;
    unsigned m = (1u << CAND) - 1;
    for (int t = threadIdx.x; t < p.Np; t += blockDim.x) {
      const int64_t node = e * p.Np + t;
      const double mj = p.MJ[node];
      for (int c = 0; c < CAND; ++c)
        if (wp[t] * candidate(J0, c) != mj) m &= ~(1u << c);
      good = good && 1 / mj == p.MJI[node];
      for (int a = 0; a < dim; ++a)
        for (int c = 0; c < dim; ++c) {
          const int64_t at = (int64_t)(a + dim * c) * p.Ntot;
          good = good && p.g[at + node] == (a == c ? p.g[at + e * p.Np] : 0.0);
        }
    }
    atomicAnd(&mJ, m);
    double fJ0[3] = {1, 1, 1};
    unsigned mf[3] = {(1u << CAND) - 1, (1u << CAND) - 1, (1u << CAND) - 1};
    for (int r = 0; r < dim; ++r) {
      fJ0[r] = p.faceMJ[e * p.Nfp + 2 * r * p.Nfpf] / wf[0];
      good = good && fJ0[r] > 1e-300 && fJ0[r] < 1e300;
    }
    for (int f = threadIdx.x; f < p.Nfp; f += blockDim.x) {
      const int face = f / p.Nfpf, fp = f - face * p.Nfpf, r = face >> 1, side = face & 1;
      const int64_t jj = e * p.Nfp + f;
      for (int c = 0; c < CAND; ++c)
        if (wf[fp] * candidate(fJ0[r], c) != p.faceMJ[jj]) mf[r] &= ~(1u << c);
      for (int d = 0; d < dim; ++d)
        good = good && p.normal[d * p.NF + jj] == (d == r ? (side ? 1.0 : -1.0) : 0.0);
      if (p.bctag[e * (2 * dim) + face] == 0) {
        // the same point of the opposite face of one element
        int st = 1, pos = 0, rem = fp;
        for (int d = 0; d < dim; ++d) {
          if (d == r) {
            pos += (side ? 0 : p.Nq - 1) * st;
          } else {
            pos += (rem % p.Nq) * st;
            rem /= p.Nq;
          }
          st *= p.Nq;
        }
        const int64_t en = p.faceix_p[e * p.Nfp + face * p.Nfpf] / p.Np;
        good = good && p.faceix_p[jj] == en * p.Np + pos;
      }
    }
    for (int r = 0; r < dim; ++r) atomicAnd(&mF[r], mf[r]);
    if (!good) ok = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
      bool box = ok && mJ;
      for (int r = 0; r < dim; ++r) box = box && mF[r];
      if (box) {
        double g[3], fJ[3];
        int32_t nb[6];
        for (int r = 0; r < dim; ++r) {
          g[r] = p.g[(int64_t)(r + dim * r) * p.Ntot + e * p.Np];
          fJ[r] = candidate(fJ0[r], pick(mF[r]));
        }
        const double J = candidate(J0, pick(mJ));
        // (a box's own are a few roundings apart)
        if (lift)
          for (int r = 0; r < dim; ++r)
            if (!(fabs(g[r] * J - fJ[r]) <= 64 * 2.220446049250313e-16 * fJ[r])) *bad = 1;
        for (int f = 0; f < 2 * dim; ++f) {
          const int tag = p.bctag[e * (2 * dim) + f];
          nb[f] = tag ? -tag : (int32_t)(p.faceix_p[e * p.Nfp + f * p.Nfpf] / p.Np);
        }
        store_record(rec + e * bytes, dim, g, J, fJ, nb);
      } else {
        *bad = 1;
      }
    }
    __syncthreads();
  }
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

int dg_box(atm_dg* dg, const atm_dg_desc* d) {
  DevDG& p = dg->dev;
  Resolved r;
  if (!box_kernels(dg, d, &r)) return ATM_OK;
  atm_ctx* ctx = dg->ctx;
  const int dim = dg->dim, Nq = dg->Nq, Np = dg->Np;
  double w[8];
  lgl_weights(Nq, w);
  std::vector<double> tab = box_tables(dim, Nq, w);
  tab.push_back(0.0);  // the flag that box_detect_kernel raises
  const size_t bytes = box_elem_bytes(dim);
  const size_t head = (tab.size() * sizeof(double) + 255) / 256 * 256;
  void* mem = nullptr;
  HIPCHK(ctx, hipMalloc(&mem, head + bytes * (size_t)p.K));
  double* dtab = static_cast<double*>(mem);
  int32_t* bad = reinterpret_cast<int32_t*>(dtab + tab.size() - 1);
  char* rec = static_cast<char*>(mem) + head;
  hipStream_t s = stream_of(ctx);
  int32_t host_bad = 1;
  hipError_t e = hipMemcpy(mem, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(box_detect_kernel, dim3(p.K < 65536 ? p.K : 65536), dim3(Np > 128 ? 256 : 64), 0, s, p, dim,
                       dtab + Nq, dtab + Nq + Np, rec, (int)bytes, box_lift(d), bad);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e == hipSuccess) e = hipMemcpy(&host_bad, bad, sizeof(int32_t), hipMemcpyDeviceToHost);
  if (e != hipSuccess || host_bad) {
    hipFree(mem);
    return e == hipSuccess ? ATM_OK : hipfail(ctx, e, "box element detection");
  }
  dg->allocs.push_back(mem);
  dg->dev_bytes += head + bytes * (size_t)p.K;
  dg_use_box(dg, r, rec, dtab);
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
