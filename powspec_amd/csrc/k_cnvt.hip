// k_cnvt.hip -- survey coordinate conversion on gfx950 (src/cnvt_coord.c):
// (RA, Dec, redshift) -> comoving Cartesian coordinates, FP64.
#include <float.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include <hip/hip_runtime.h>

#include "powspec_hip.h"
#include "psh_internal.h"

namespace {

constexpr int kMinOrder = 4, kMaxOrder = 32;   // math/legauss.h:40-41
constexpr int kNumZ = 128;                     // POWSPEC_INT_NUM_ZSP (src/define.h:93)
constexpr double kCH = 299792.458 * 0.01;      // c / (100 km/s/Mpc), Mpc/h
constexpr double kDeg = M_PI / 180;

// Gauss-Legendre rule of order n: the n/2 positive abscissas with weights and
// the weight of x = 0 for odd n, from Newton's iteration on P_n in long
// double (P_n, P_n' by the three-term recurrence).
struct Rule {
  double x[kMaxOrder / 2 + 1], w[kMaxOrder / 2 + 1], w0;
};

Rule legauss_rule(int n) {
  Rule r{};
  auto legendre = [n](long double t, long double &pn, long double &pn1) {
    long double a = 1, b = t;
    for (int j = 2; j <= n; j++) {
      long double c = ((2 * j - 1) * t * b - (j - 1) * a) / j;
      a = b;
      b = c;
    }
    pn = b;
    pn1 = a;
  };
  for (int k = 0; k < n / 2; k++) {
    long double t = cosl(M_PI * (k + 0.75L) / (n + 0.5L)), pn, pn1;
    for (int it = 0; it < 100; it++) {
      legendre(t, pn, pn1);
      long double dt = pn / (n * (t * pn - pn1) / (t * t - 1));
      t -= dt;
      if (fabsl(dt) < 1e-19L) break;
    }
    legendre(t, pn, pn1);
    long double dp = n * (t * pn - pn1) / (t * t - 1);
    r.x[k] = (double)t;
    r.w[k] = (double)(2 / ((1 - t * t) * dp * dp));
  }
  if (n & 1) {
    long double pn, pn1;
    legendre(0, pn, pn1);
    long double dp = n * pn1;
    r.w0 = (double)(2 / (dp * dp));
  }
  return r;
}

struct Cosmo {
  double om, ol, ok, widx;
};

// E(z)^2 with the terms in the reference's order (src/cnvt_coord.c:241-252)
__host__ __device__ inline double efunc2(const Cosmo &c, double z) {
#pragma clang fp contract(off)
  double z1 = z + 1;
  double z2 = z1 * z1;
  double d = c.om * z2 * z1;
  if (c.ok) d += c.ok * z2;
  if (c.widx) d += c.ol * pow(z1, c.widx);
  else d += c.ol;
  return d;
}

struct RuleDev {
  int n;
  double x[kMaxOrder / 2 + 1], w[kMaxOrder / 2 + 1], w0;
};

// The order search compares distances of successive orders: written without
// fused operations, host and device round alike (but for pow, see
// psh_cnvt_device) and settle on the same order.
__host__ __device__ inline double cmvdist(const Cosmo &c, const RuleDev &r, double z) {
#pragma clang fp contract(off)
  auto f = [&](double t) {
#pragma clang fp contract(off)
    return kCH / sqrt(efunc2(c, t));
  };
  double zp = z * 0.5, sum = 0;
  for (int k = 0; k < r.n / 2; k++)
    sum += r.w[k] * (f(zp * (1 + r.x[k])) + f(zp * (1 - r.x[k])));
  if (r.n & 1) sum += r.w0 * f(zp);
  return sum * zp;
}

RuleDev rule_dev(int n) {
  Rule r = legauss_rule(n);
  RuleDev d{};
  d.n = n;
  memcpy(d.x, r.x, sizeof d.x);
  memcpy(d.w, r.w, sizeof d.w);
  d.w0 = r.w0;
  return d;
}

__device__ inline void to_cartesian(double *p, double dist) {
  const double ra = p[0] * kDeg, dec = p[1] * kDeg;
  double sr, cr, sd, cd;   // (one argument reduction for both)
  sincos(ra, &sr, &cr);
  sincos(dec, &sd, &cd);
  p[0] = dist * cd * cr;
  p[1] = dist * cd * sr;
  p[2] = dist * sd;
}

// Workspace of the integrated conversion on the device.
struct CnvtDev {
  double zmin, zmax;   // of the arrays seen so far
  int order;           // > 0 found; 0 nothing to convert; -1 error
  RuleDev rules[kMaxOrder + 2 - kMinOrder];   // orders kMinOrder..kMaxOrder + 1
};

// 1 / E(z): the distance integral with reciprocal square roots, whose
// rounding (1 ulp against 1/2 + 1/2 of a root and a division) is far below
// the quadrature's error, and a third of their instructions: 2e7 records at
// order 5 took 377 us, bound by FP64 arithmetic, now 286 us; moving their
// 1.28 GB takes 266 us.
template <bool K, bool W>
__device__ inline double distance(const Cosmo &c, const RuleDev &r, double z) {
  auto f = [&](double t) -> double {
    const double z1 = t + 1, z2 = z1 * z1;
    double d = W ? c.ol * pow(z1, c.widx) : c.ol;
    d = __builtin_fma(c.om * z2, z1, d);
    if (K) d = __builtin_fma(c.ok, z2, d);
    return rsqrt(d);
  };
  const double zp = z * 0.5;
  double sum = 0;
  for (int k = 0; k < r.n / 2; k++)
    sum = __builtin_fma(r.w[k], f(__builtin_fma(zp, r.x[k], zp)) + f(__builtin_fma(-zp, r.x[k], zp)),
                        sum);
  if (r.n & 1) sum = __builtin_fma(r.w0, f(zp), sum);
  return sum * (zp * kCH);
}

template <bool K, bool W>
__global__ void __launch_bounds__(256)
integr_kernel(double *d, size_t n, Cosmo c, const CnvtDev *ws) {
  const int order = ws->order;
  if (order <= 0) return;
  const RuleDev &r = ws->rules[order - kMinOrder];
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    double *p = d + 4 * i;
    to_cartesian(p, distance<K, W>(c, r, p[2]));
  }
}

// Smallest order at which the integral to z has converged
// (src/cnvt_coord.c:306-341): orders are tried from kMinOrder up; the test
// reaches order kMaxOrder + 1 before it gives up (the reference reads that
// rule past the end of its table; here it is computed), -1 when that does not
// converge either.
__host__ __device__ inline int order_at(const Cosmo &c, const RuleDev *rules, double err,
                                        double z) {
#pragma clang fp contract(off)
  double oint, nint = 0;
  int n = kMinOrder - 1;
  do {
    if (n > kMaxOrder) return -1;
    oint = nint;
    ++n;
    nint = cmvdist(c, rules[n - kMinOrder], z);
  } while (fabs(nint - oint) > nint * err);
  return n;
}

// i-th of the kNumZ redshifts of the convergence test
__host__ __device__ inline double test_z(double zmin, double zmax, int i) {
#pragma clang fp contract(off)
  return zmin + i * (zmax - zmin) / (kNumZ - 1);
}

// The order of a redshift range: the largest of the test redshifts' (-1 when
// one of them does not converge).
int choose_order(const Cosmo &c, const RuleDev *rules, double err, double zmin, double zmax) {
  int order = 0;
  for (int i = 0; i < kNumZ; i++) {
    const int n = order_at(c, rules, err, test_z(zmin, zmax, i));
    if (n < 0) return -1;
    if (order < n) order = n;
  }
  return order;
}

// Takes the redshift bounds of one array's blocks into ws; with `last`, finds
// the order, one test redshift per thread.  One workgroup.  (On the host the
// same search, the copies to and from it and the tables of its 30 rules, made
// anew on each call, took 330 us.)
__global__ void __launch_bounds__(256)
order_kernel(CnvtDev *ws, const double *__restrict__ part, int blocks, int first, int last,
             Cosmo c, double err, double *__restrict__ hout) {
  __shared__ double mn[256], mx[256];
  __shared__ int worst;
  const int t = threadIdx.x;
  double a = DBL_MAX, b = -DBL_MAX;
  for (int i = t; i < blocks; i += 256) {
    a = fmin(a, part[PSH_BOUNDS_STRIDE * i + 2]);
    b = fmax(b, part[PSH_BOUNDS_STRIDE * i + 5]);
  }
  mn[t] = a;
  mx[t] = b;
  if (t == 0) worst = 0;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (t < k) {
      mn[t] = fmin(mn[t], mn[t + k]);
      mx[t] = fmax(mx[t], mx[t + k]);
    }
    __syncthreads();
  }
  double zmin = mn[0], zmax = mx[0];
  if (!first) {
    zmin = fmin(zmin, ws->zmin);
    zmax = fmax(zmax, ws->zmax);
  }
  __syncthreads();   // (every thread has read the earlier bounds)
  const bool any = zmin <= zmax && zmin >= 0;   // something to convert, no negative redshift
  if (last && any && t < kNumZ) {
    const int n = order_at(c, ws->rules, err, test_z(zmin, zmax, t));
    atomicMax(&worst, n < 0 ? kMaxOrder + 2 : n);
  }
  __syncthreads();
  if (t == 0) {
    ws->zmin = zmin;
    ws->zmax = zmax;
    if (last) {
      const int order = zmin > zmax ? 0 : (!any || worst > kMaxOrder + 1) ? -1 : worst;
      ws->order = order;
      hout[0] = zmin;
      hout[1] = zmax;
      hout[2] = (double)order;
    }
  }
}

// Natural cubic spline with the reference's interval search
// (src/cnvt_coord.c:97-111): HUGE_VAL outside [zs[0], zs[n-1]).
__global__ void __launch_bounds__(256) interp_kernel(double *d, size_t n, const double *zs,
                                                     const double *ds, const double *ypp,
                                                     size_t nsp) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    double *p = d + 4 * i;
    const double z = p[2];
    double dist = HUGE_VAL;
    if (z >= zs[0] && z < zs[nsp - 1]) {
      size_t lo = 0, hi = nsp - 1;
      while (hi - lo > 1) {
        const size_t mid = (lo + hi) >> 1;
        if (zs[mid] <= z) lo = mid;
        else hi = mid;
      }
      const double b = zs[lo + 1] - zs[lo], a = z - zs[lo], e = zs[lo + 1] - z;
      dist = (a * ds[lo + 1] + e * ds[lo] +
              ((a * a - b * b) * a * ypp[lo + 1] + (e * e - b * b) * e * ypp[lo]) / 6) / b;
    }
    to_cartesian(p, dist);
  }
}

// Second derivatives of the natural spline (zero at both ends).
std::vector<double> spline_ypp(const double *x, const double *y, size_t n) {
  std::vector<double> ypp(n, 0.0), c(n, 0.0);
  for (size_t j = 1; j + 1 < n; j++) {
    const double h0 = x[j] - x[j - 1], h1 = x[j + 1] - x[j];
    const double rhs = 6 * ((y[j + 1] - y[j]) / h1 - (y[j] - y[j - 1]) / h0);
    const double piv = 2 * (h0 + h1) - h0 * c[j - 1];
    ypp[j] = (rhs - h0 * ypp[j - 1]) / piv;
    c[j] = h1 / piv;
  }
  for (size_t j = n - 1; j-- > 0;) ypp[j] -= c[j] * ypp[j + 1];
  return ypp;
}

unsigned blocks_for(size_t n) {
  size_t b = (n + 255) / 256;
  if (b > 8192) b = 8192;
  return (unsigned)(b ? b : 1);
}

// Workspace of one call: the device block, per-block bounds and the pinned
// results.  Calls take one and give it back when their work is done; at most
// kKeep of them stay for later calls.
constexpr int kBoundsBlocks = 1024;
struct Workspace {
  int device = -1;
  CnvtDev *dev = nullptr;
  double *part = nullptr;
  double *hout = nullptr;   // zmin, zmax, order
};

void free_workspace(Workspace &w) {
  if (w.dev) (void)hipFree(w.dev);
  if (w.part) (void)hipFree(w.part);
  if (w.hout) (void)hipHostFree(w.hout);
  w = Workspace{};
}

struct Workspaces {
  static constexpr size_t kKeep = 4;
  std::mutex m;
  std::vector<Workspace> idle;

  bool take(const std::vector<RuleDev> &rules, Workspace &w) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    {
      std::lock_guard<std::mutex> lock(m);
      for (size_t i = 0; i < idle.size(); i++)
        if (idle[i].device == dev) {
          w = idle[i];
          idle.erase(idle.begin() + (long)i);
          return true;
        }
    }
    w.device = dev;
    if (psh_malloc(&w.dev, sizeof(CnvtDev)) == hipSuccess &&
        psh_malloc(&w.part, sizeof(double) * PSH_BOUNDS_STRIDE * kBoundsBlocks) ==
            hipSuccess &&
        hipHostMalloc((void **)&w.hout, 3 * sizeof(double), hipHostMallocDefault) == hipSuccess &&
        hipMemcpy(w.dev->rules, rules.data(), sizeof(w.dev->rules), hipMemcpyHostToDevice) ==
            hipSuccess)
      return true;
    (void)hipGetLastError();   // (of the host allocation or the copy)
    free_workspace(w);
    return false;
  }
  void give(Workspace &w) {
    {
      std::lock_guard<std::mutex> lock(m);
      if (idle.size() < kKeep) {
        idle.push_back(w);
        return;
      }
    }
    free_workspace(w);
  }
};

// (never destroyed: the HIP runtime may end before static destructors run)
Workspaces &workspaces() {
  static Workspaces *w = new Workspaces;
  return *w;
}

// The quadrature rules of the orders kMinOrder..kMaxOrder + 1.
const std::vector<RuleDev> &all_rules() {
  static const std::vector<RuleDev> rules = [] {
    std::vector<RuleDev> r;
    for (int n = kMinOrder; n <= kMaxOrder + 1; n++) r.push_back(rule_dev(n));
    return r;
  }();
  return rules;
}

// Redshift range of everything to be converted (src/cnvt_coord.c:138-226),
// its order and the conversion, on one stream with one wait at the end.
int integrate(const psh_cnvt *cv, const Cosmo &c, psh_data *const *d_data, const size_t *n,
              int narr, const Workspace &w, hipStream_t s, int *order_out) {
  int lasta = -1;
  for (int a = 0; a < narr; a++)
    if (n[a]) lasta = a;
  if (order_out) *order_out = 0;
  if (lasta < 0) return PSH_OK;   // nothing to convert
  bool first = true;
  for (int a = 0; a <= lasta; a++) {
    if (!n[a]) continue;
    int blocks = (int)std::min<size_t>((n[a] + 255) / 256, kBoundsBlocks);
    if (psh_coord_bounds((const double *)d_data[a], n[a], w.part, blocks, s) != hipSuccess)
      return PSH_ERR_DEVICE;
    hipLaunchKernelGGL(order_kernel, dim3(1), dim3(256), 0, s, w.dev, w.part, blocks, (int)first,
                       (int)(a == lasta), c, cv->ecdst, w.hout);
    if (hipGetLastError() != hipSuccess) return PSH_ERR_DEVICE;
    first = false;
  }
  if (c.widx) {
    // pow of the host and of the device may differ in the last bit, and the
    // order with it where a test is that close: the host decides
    if (hipStreamSynchronize(s) != hipSuccess) return PSH_ERR_DEVICE;
    int order = (int)w.hout[2];
    if (w.hout[0] <= w.hout[1] && w.hout[0] >= 0) {
      order = choose_order(c, all_rules().data(), cv->ecdst, w.hout[0], w.hout[1]);
      if (order < 0) return PSH_ERR_CNVT;
      if (hipMemcpy(&w.dev->order, &order, sizeof order, hipMemcpyHostToDevice) != hipSuccess)
        return PSH_ERR_DEVICE;
      w.hout[2] = (double)order;
    }
  }
  for (int a = 0; a <= lasta; a++) {
    if (!n[a]) continue;
    auto go = [&](auto k, auto x) {
      hipLaunchKernelGGL((integr_kernel<decltype(k)::value, decltype(x)::value>),
                         dim3(blocks_for(n[a])), dim3(256), 0, s, (double *)d_data[a], n[a], c,
                         w.dev);
    };
    if (c.ok) c.widx ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
    else c.widx ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
    if (hipGetLastError() != hipSuccess) return PSH_ERR_DEVICE;
  }
  if (hipStreamSynchronize(s) != hipSuccess) return PSH_ERR_DEVICE;
  const int order = (int)w.hout[2];
  if (order < 0) return PSH_ERR_CNVT;   // negative redshift, or no convergence
  if (order_out) *order_out = order;
  return PSH_OK;
}

}  // namespace

extern "C" int psh_cnvt_device(const psh_cnvt *cv, psh_data *const *d_data, const size_t *n,
                               int narr, int *order_out) {
  if (!cv || narr < 0 || (narr && (!d_data || !n))) return PSH_ERR_ARG;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return PSH_ERR_DEVICE;
  hipStream_t s = nullptr;
  const Cosmo c{cv->omega_m, cv->omega_l, cv->omega_k,
                cv->eos_w == -1 ? 0.0 : 3 * (1 + cv->eos_w)};   // src/cnvt_coord.c:498
  if (cv->zsp) {
    if (!cv->dsp || cv->nsp < 2) return PSH_ERR_ARG;
    std::vector<double> ypp = spline_ypp(cv->zsp, cv->dsp, cv->nsp);
    double *tab = nullptr;
    if (psh_malloc(&tab, sizeof(double) * 3 * cv->nsp) != hipSuccess) return PSH_ERR_MEMORY;
    bool ok = hipMemcpy(tab, cv->zsp, sizeof(double) * cv->nsp, hipMemcpyHostToDevice) ==
                  hipSuccess &&
              hipMemcpy(tab + cv->nsp, cv->dsp, sizeof(double) * cv->nsp,
                        hipMemcpyHostToDevice) == hipSuccess &&
              hipMemcpy(tab + 2 * cv->nsp, ypp.data(), sizeof(double) * cv->nsp,
                        hipMemcpyHostToDevice) == hipSuccess;
    for (int a = 0; ok && a < narr; a++) {
      if (!n[a]) continue;
      hipLaunchKernelGGL(interp_kernel, dim3(blocks_for(n[a])), dim3(256), 0, s,
                         (double *)d_data[a], n[a], tab, tab + cv->nsp, tab + 2 * cv->nsp,
                         cv->nsp);
      ok = hipGetLastError() == hipSuccess;
    }
    ok = ok && hipStreamSynchronize(s) == hipSuccess;
    (void)hipFree(tab);
    if (order_out) *order_out = 0;
    return ok ? PSH_OK : PSH_ERR_DEVICE;
  }
  Workspace w;
  if (!workspaces().take(all_rules(), w)) return PSH_ERR_MEMORY;
  int order = 0;
  const int rc = integrate(cv, c, d_data, n, narr, w, s, &order);
  // an error may have left work in flight that writes the workspace
  if (rc == PSH_ERR_DEVICE) (void)hipStreamSynchronize(s);
  workspaces().give(w);
  if (rc == PSH_OK && order_out) *order_out = order;
  return rc;
}

extern "C" int psh_cnvt_coord(const psh_cnvt *cv, psh_cata *cat) {
  if (!cv || !cat) return PSH_ERR_ARG;
  std::vector<psh_data *> host, dev;
  std::vector<size_t> cnt;
  for (int i = 0; i < cat->num && i < 2; i++) {
    if (cv->dcnvt[i] && cat->ndata[i]) {
      host.push_back(cat->data[i]);
      cnt.push_back(cat->ndata[i]);
    }
    if (cv->rcnvt[i] && cat->rand && cat->nrand && cat->nrand[i]) {
      host.push_back(cat->rand[i]);
      cnt.push_back(cat->nrand[i]);
    }
  }
  int rc = PSH_OK;
  for (size_t a = 0; a < host.size(); a++) {
    psh_data *d = nullptr;
    if (psh_malloc(&d, sizeof(psh_data) * cnt[a]) != hipSuccess ||
        hipMemcpy(d, host[a], sizeof(psh_data) * cnt[a], hipMemcpyHostToDevice) !=
            hipSuccess) {
      if (d) (void)hipFree(d);
      rc = PSH_ERR_DEVICE;
      break;
    }
    dev.push_back(d);
  }
  if (rc == PSH_OK) rc = psh_cnvt_device(cv, dev.data(), cnt.data(), (int)dev.size(), nullptr);
  for (size_t a = 0; a < dev.size(); a++) {
    if (rc == PSH_OK &&
        hipMemcpy(host[a], dev[a], sizeof(psh_data) * cnt[a], hipMemcpyDeviceToHost) !=
            hipSuccess)
      rc = PSH_ERR_DEVICE;
    (void)hipFree(dev[a]);
  }
  return rc;
}
