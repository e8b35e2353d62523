// The lockstep reductions against sums on the host, and the Krylov solvers'
// iterate-only switch against the solve that also forms its last residual.
//
//  * bdots_dev (inner products and norm) and bbicg_xr_dots (the reductions in its
//    update pass), FP64 and FP32 with paired and unpaired loads, with rhs whose
//    elements lie within, across and beyond a workgroup's 256 threads: every sum
//    within 1e-12 of the host's, relative to the norms (FP64 sums of 1e5 terms and
//    more, 1e-14; one run of threads left out or counted twice is 1e-3 or more).
//  * Gmres and BGmres: the iterates must agree to the bit, and the residual that the
//    recurrence estimates with the true one to its rounding.
//
// Prints "ALL PASSED" and exits 0 on success.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "bblas.hpp"
#include "bkrylov.hpp"
#include "blas.hpp"
#include "krylov.hpp"

using namespace mgc;

namespace {

int g_fail = 0;

#define HIPOK(x)                                                               \
  do {                                                                         \
    hipError_t e_ = (x);                                                       \
    if (e_ != hipSuccess) {                                                    \
      std::printf("HIP error %s at %s:%d\n", hipGetErrorString(e_), __FILE__, \
                  __LINE__);                                                   \
      std::exit(2);                                                            \
    }                                                                          \
  } while (0)

template <typename T> struct Dev {
  T* p = nullptr;
  size_t n = 0;
  explicit Dev(size_t count) : n(count) { HIPOK(hipMalloc(&p, count * sizeof(T))); }
  explicit Dev(const std::vector<T>& h) : Dev(h.size()) { put(h); }
  ~Dev() { (void)hipFree(p); }
  Dev(const Dev&) = delete;
  Dev& operator=(const Dev&) = delete;
  void put(const std::vector<T>& h) {
    HIPOK(hipMemcpy(p, h.data(), n * sizeof(T), hipMemcpyHostToDevice));
  }
  std::vector<T> get() const {
    std::vector<T> h(n);
    HIPOK(hipMemcpy(h.data(), p, n * sizeof(T), hipMemcpyDeviceToHost));
    return h;
  }
};

template <typename R> std::vector<cplx<R>> random_vec(size_t n, uint64_t seed) {
  std::mt19937_64 g(seed);
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  std::vector<cplx<R>> v(n);
  for (auto& z : v) z = {(R)u(g), (R)u(g)};
  return v;
}

void report(const char* what, const char* prec, const char* shape, bool ok) {
  std::printf("%-14s %-4s %s : %s\n", what, prec, shape, ok ? "ok" : "FAIL");
  std::fflush(stdout);
  if (!ok) ++g_fail;
}

// per-rhs <a, b> on the host
template <typename R>
std::vector<cplx<double>> host_dots(const cplx<R>* a, const cplx<R>* b, const BShape& sh) {
  std::vector<cplx<double>> o(sh.nrhs, cplx<double>{0.0, 0.0});
  for (size_t i = 0; i < sh.n; ++i) {
    cplx<double>& t = o[(i % sh.cols()) / sh.dof];
    const double ar = a[i].re, ai = a[i].im, br = b[i].re, bi = b[i].im;
    t.re += ar * br + ai * bi;
    t.im += ar * bi - ai * br;
  }
  return o;
}

bool near(cplx<double> got, cplx<double> want, double aa, double bb) {
  return std::hypot(got.re - want.re, got.im - want.im) <= 1e-12 * std::sqrt(aa * bb);
}

template <typename R>
void dots_case(BBlas& b, const char* prec, size_t sites, int nrhs, int dof, int k, size_t pad,
               uint64_t seed) {
  BShape sh;
  sh.nrhs = nrhs;
  sh.dof = dof;
  sh.n = sites * (size_t)sh.cols();
  const size_t ldv = sh.n + pad;
  const auto V = random_vec<R>((size_t)k * ldv, seed), w = random_vec<R>(sh.n, seed + 1);
  Dev<cplx<R>> dV(V), dw(w);
  Dev<cplx<double>> d((size_t)(k + 1) * nrhs);
  bdots_dev<R>(b, dV.p, ldv, k, dw.p, sh, true, d.p);
  HIPOK(hipStreamSynchronize(b.s));
  const auto got = d.get();
  const auto ww = host_dots<R>(w.data(), w.data(), sh);
  bool ok = true;
  for (int j = 0; j < k; ++j) {
    const cplx<R>* v = V.data() + (size_t)j * ldv;
    const auto vw = host_dots<R>(v, w.data(), sh), vv = host_dots<R>(v, v, sh);
    for (int r = 0; r < nrhs; ++r) ok &= near(got[(size_t)j * nrhs + r], vw[r], vv[r].re, ww[r].re);
  }
  for (int r = 0; r < nrhs; ++r)
    ok &= near({got[(size_t)k * nrhs + r].re, 0.0}, {ww[r].re, 0.0}, ww[r].re, ww[r].re);
  char s[96];
  std::snprintf(s, sizeof s, "sites=%zu nrhs=%d dof=%d k=%d", sites, nrhs, dof, k);
  report("bdots", prec, s, ok);
}

template <typename R>
void xr_case(BBlas& b, const char* prec, size_t sites, int nrhs, int dof, uint64_t seed) {
  BShape sh;
  sh.nrhs = nrhs;
  sh.dof = dof;
  sh.n = sites * (size_t)sh.cols();
  Dev<cplx<R>> p(random_vec<R>(sh.n, seed)), s(random_vec<R>(sh.n, seed + 1)),
      t(random_vec<R>(sh.n, seed + 2)), x(random_vec<R>(sh.n, seed + 3)),
      r(random_vec<R>(sh.n, seed + 4));
  const auto rh = random_vec<R>(sh.n, seed + 5);
  Dev<cplx<R>> drh(rh);
  std::vector<cplx<double>> c(random_vec<double>((size_t)3 * nrhs, seed + 6));
  const int stopped = nrhs > 2 ? nrhs / 2 : -1;
  for (int q = 0; q < nrhs; ++q) c[(size_t)2 * nrhs + q] = {q == stopped ? 0.0 : 1.0, 0.0};
  Dev<cplx<double>> d((size_t)2 * nrhs);
  bbicg_xr_dots<R>(b, c.data(), p.p, s.p, t.p, drh.p, x.p, r.p, sh, d.p);
  HIPOK(hipStreamSynchronize(b.s));
  const auto got = d.get();
  const auto rn = r.get();  // the updated residual
  const auto rr = host_dots<R>(rn.data(), rn.data(), sh);
  const auto hr = host_dots<R>(rh.data(), rn.data(), sh), hh = host_dots<R>(rh.data(), rh.data(), sh);
  bool ok = true;
  for (int q = 0; q < nrhs; ++q) {
    if (q == stopped) {
      ok &= got[q].re == 0.0 && got[(size_t)nrhs + q].re == 0.0 && got[(size_t)nrhs + q].im == 0.0;
      continue;
    }
    ok &= near({got[q].re, 0.0}, {rr[q].re, 0.0}, rr[q].re, rr[q].re);
    ok &= near(got[(size_t)nrhs + q], hr[q], hh[q].re, rr[q].re);
  }
  char m[96];
  std::snprintf(m, sizeof m, "sites=%zu nrhs=%d dof=%d", sites, nrhs, dof);
  report("bbicg_xr_dots", prec, m, ok);
}

// y_i = d_i x_i + (0.3 + 0.1 i) x_(i + stride mod n): well conditioned, not normal
template <typename R>
__global__ void k_test_op(const cplx<R>* x, cplx<R>* y, size_t n, size_t stride) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const cplx<R> a = x[i], b = x[(i + stride) % n];
    const R d = R(1) + R(0.5) * R((i * 2654435761u % 1024) / 1024.0);
    y[i] = {d * a.re + R(0.3) * b.re - R(0.1) * b.im, d * a.im + R(0.3) * b.im + R(0.1) * b.re};
  }
}
template <typename R> struct TestOp : LinOp<R> {
  void apply(const cplx<R>* in, cplx<R>* out, hipStream_t s) override {
    k_test_op<R><<<256, 256, 0, s>>>(in, out, this->n, 1);
  }
};
template <typename R> struct BTestOp : BLinOp<R> {
  void apply(const cplx<R>* in, cplx<R>* out, hipStream_t s) override {
    k_test_op<R><<<256, 256, 0, s>>>(in, out, this->sh.n, this->sh.cols());  // within an rhs
  }
};

template <typename T> bool same_bits(const std::vector<T>& a, const std::vector<T>& b) {
  return a.size() == b.size() && std::memcmp(a.data(), b.data(), a.size() * sizeof(T)) == 0;
}

template <typename R>
void iterate_case(hipStream_t s, const char* prec, int m, int maxit, double tol, bool x_zero,
                  bool flexible, double eta) {
  const size_t n = 40000;
  Blas bl(s);
  TestOp<R> A;
  A.n = n;
  Dev<cplx<R>> b(random_vec<R>(n, 7)), x(n);
  const auto x0 = random_vec<R>(n, 8);
  std::vector<cplx<R>> xs[2];
  KrylovStats st[2];
  for (int on = 0; on < 2; ++on) {
    Gmres<R> g(n, m, flexible);
    g.set_reorth_eta(eta);
    g.set_iterate_only(on);
    x.put(x0);
    st[on] = g.solve(bl, A, nullptr, b.p, x.p, x_zero, tol, maxit);
    HIPOK(hipStreamSynchronize(s));
    xs[on] = x.get();
  }
  const double slack = sizeof(R) == 8 ? 1e-9 : 1e-3;
  const bool ok = same_bits(xs[0], xs[1]) && st[0].iters == st[1].iters &&
                  std::fabs(st[0].rel_res - st[1].rel_res) <= slack;
  char t[128];
  std::snprintf(t, sizeof t, "m=%d maxit=%d tol=%g x0=%d flexible=%d eta=%g iters=%d", m, maxit,
                tol, !x_zero, flexible, eta, st[0].iters);
  report("Gmres", prec, t, ok);
}

template <typename R>
void biterate_case(hipStream_t s, const char* prec, int m, int maxit, double tol, bool x_zero,
                   bool flexible, double eta) {
  BShape sh;
  sh.nrhs = 5;
  sh.dof = 12;
  sh.n = (size_t)1024 * sh.cols();
  BBlas bl(s);
  BTestOp<R> A;
  A.sh = sh;
  auto hb = random_vec<R>(sh.n, 9);
  for (size_t i = 0; i < sh.n; ++i)  // rhs 3 is zero, rhs 1 small
    if ((i % sh.cols()) / sh.dof == 3) hb[i] = {R(0), R(0)};
    else if ((i % sh.cols()) / sh.dof == 1) hb[i] = {R(1e-3) * hb[i].re, R(1e-3) * hb[i].im};
  Dev<cplx<R>> b(hb), x(sh.n);
  const auto x0 = random_vec<R>(sh.n, 10);
  std::vector<cplx<R>> xs[2];
  BKrylovStats st[2];
  for (int on = 0; on < 2; ++on) {
    BGmres<R> g(sh, m, flexible);
    g.set_reorth_eta(eta);
    g.set_iterate_only(on);
    x.put(x0);
    st[on] = g.solve(bl, A, nullptr, b.p, x.p, x_zero, tol, maxit);
    HIPOK(hipStreamSynchronize(s));
    xs[on] = x.get();
  }
  bool ok = same_bits(xs[0], xs[1]) && st[0].iters == st[1].iters;
  const double slack = sizeof(R) == 8 ? 1e-9 : 1e-3;
  for (int r = 0; r < sh.nrhs; ++r)  // (rhs 1 starts far from its solution where x0 is not zero)
    ok &= std::fabs(st[0].rel_res[r] - st[1].rel_res[r]) <= slack * (1.0 + st[0].rel_res[r]) ||
          (r == 1 && !x_zero);
  char t[128];
  std::snprintf(t, sizeof t, "m=%d maxit=%d tol=%g x0=%d flexible=%d eta=%g iters=%d", m, maxit,
                tol, !x_zero, flexible, eta, st[0].iters);
  report("BGmres", prec, t, ok);
}

}  // namespace

int main() {
  try {
    hipStream_t s;
    HIPOK(hipStreamCreate(&s));
    {
      BBlas b(s);
      // columns per site below, at, above and no divisor of 256; dof above 256; one
      // rhs; odd dof (unpaired FP32 loads)
      const int shapes[][2] = {{12, 12}, {5, 3}, {7, 13}, {2, 64}, {8, 32},  {4, 64}, {3, 100},
                               {33, 16}, {64, 4}, {1, 12}, {1, 300}, {2, 300}, {3, 257}};
      uint64_t seed = 5000;
      for (const auto& q : shapes) {
        const size_t sites = 200000 / ((size_t)q[0] * q[1]) + 1;
        for (int k : {0, 3, 9}) {
          dots_case<double>(b, "f64", sites, q[0], q[1], k, 0, seed += 10);
          dots_case<float>(b, "f32", sites, q[0], q[1], k, 0, seed += 10);
        }
        dots_case<float>(b, "f32", sites, q[0], q[1], 3, 1, seed += 10);  // odd rows: unpaired
        dots_case<float>(b, "f32", 3, q[0], q[1], 3, 0, seed += 10);      // one workgroup or two
        xr_case<double>(b, "f64", sites, q[0], q[1], seed += 10);
        xr_case<float>(b, "f32", sites, q[0], q[1], seed += 10);
      }
    }
    // one cycle cut by maxit, one that fills it, restarts, a tolerance met before
    // maxit; re-orthogonalised (eta 1) or not
    for (double eta : {0.01, 1.0})
      for (bool flexible : {false, true})
        for (bool x_zero : {true, false}) {
          const struct { int m, maxit; double tol; } c[] = {
              {4, 3, 0.0}, {4, 4, 0.0}, {3, 7, 0.0}, {3, 6, 0.0}, {8, 20, 1e-2}, {1, 1, 0.0}};
          for (const auto& q : c) {
            iterate_case<double>(s, "f64", q.m, q.maxit, q.tol, x_zero, flexible, eta);
            iterate_case<float>(s, "f32", q.m, q.maxit, q.tol, x_zero, flexible, eta);
            biterate_case<double>(s, "f64", q.m, q.maxit, q.tol, x_zero, flexible, eta);
            biterate_case<float>(s, "f32", q.m, q.maxit, q.tol, x_zero, flexible, eta);
          }
        }
    HIPOK(hipStreamDestroy(s));
  } catch (const std::exception& e) {
    std::printf("exception: %s\n", e.what());
    return 3;
  }
  if (g_fail) {
    std::printf("%d case(s) FAILED\n", g_fail);
    return 1;
  }
  std::printf("ALL PASSED\n");
  return 0;
}
