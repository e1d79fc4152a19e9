// Linearized power-series Newton on real and complex multiple-double series,
// batched: one wavefront runs the whole staggered Newton method of one system
// in LDS.  The complex twins (CX) follow CPU_cmplx2_factors_houseqr,
// CPU_cmplx2_factors_qrbs, CPU_cmplx2_qrbs_head/tail/solve,
// CPU_cmplx2_linear_residue and cmplx2_row_newton_qrstep
// (Newton/cmplx2_newton_method.cpp:565) with their operation orders.
//
//   reference (host)                          here
//   CPU_dbl2_poly_evaldiff per polynomial     eval_system (slots of lanes, one
//     (Polynomials/dbl2_polynomials_host.cpp)   polynomial per slot, lane = coefficient)
//   dbl2_map_evaldiff_output, rhs = -f        read in place from the output rows
//     (Newton/dbl2_systems_host.cpp:709)
//   CPU_dbl2_factors_houseqr (Matrices/       houseqr: lane per column for the
//     dbl2_factorizations.cpp:723)              reflector products, lane per entry for updates
//   CPU_dbl2_factors_qrbs / _backward         qrbs: lane per row for Q^T b, column sweep
//     (:823, :121)                              for the back substitution
//   CPU_dbl2_qrbs_head/tail/solve             qrbs_solve: same skip rules and flags
//     (Newton/dbl2_bals_host.cpp:15,228,479)
//   CPU_dbl2_linear_residue (:548)            linear_residue
//   dbl2_row_newton_qrstep (Newton/           row_newton_kernel: the staggered loop of
//     dbl2_newton_method.cpp:429) and the       test_dbl2_row_newton (:1447-1494) in-kernel
//     staggered loop
//
// Every number is computed by the same sequence of multiple-double operations
// as the reference's host code (each lane keeps the reference's accumulation
// order for the entries it owns; lanes split only independent entries), so
// the results are bit-identical to the CPU oracle.  Lanes of one wavefront
// exchange data through LDS; within a wavefront LDS operations complete in
// program order, and wsync() keeps the compiler from moving them.
#include <vector>

#include "common.hpp"
#include "mdtypes.hpp"
#include "wave.hpp"

using namespace md;
using phc::grid_for;

namespace {

__device__ __forceinline__ void wsync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// The lanes that work on one system together: one wavefront (several of them
// in a block, each with its own system), or TW > 1 wavefronts, the whole block.
template <int TW> struct Team {
  static constexpr int N = 64 * TW;
  __device__ static __forceinline__ int id() { return TW == 1 ? (int)(threadIdx.x & 63) : (int)threadIdx.x; }
  __device__ static __forceinline__ void sync() {
    if constexpr (TW == 1) wsync();
    else __syncthreads();
  }
};

__device__ __forceinline__ double wave_fmax(double v) { return wave::max64(v); }

constexpr size_t LDS_LIMIT = 160 * 1024;

// skip thresholds of the tail solve (Newton/dbl_bals_host.cpp:199,
// dbl2_bals_host.cpp:43, dbl4_bals_host.cpp:51, dbl8_bals_host.cpp:70)
template <int K> __host__ __device__ constexpr double threshold() {
  return K == 1 ? 1.0e-15 : K == 2 ? 1.0e-28 : K == 4 ? 1.0e-56 : 1.0e-120;
}

// Real (CX = false) or complex (CX = true, K real planes then K imaginary
// planes) multiple-double numbers: the operations the Newton method needs,
// each in the order of the reference's host code of that type.
template <int K, bool CX> struct NT;
template <int K> struct NT<K, false> {
  typedef typename RealT<K>::type V;
  static constexpr int P = K;
  __device__ static V ld(const double *b, size_t m, size_t j) { return R<K>::load(b, m, j); }
  __device__ static void st(double *b, size_t m, size_t j, const V &v) { R<K>::store(b, m, j, v); }
  __device__ static V zero() { return R<K>::zero(); }
  __device__ static V one() { return R<K>::from(1.0); }
  __device__ static V add(const V &a, const V &b) { return md::add(a, b); }
  __device__ static V neg(const V &a) { return md::neg(a); }
  __device__ static V mul(const V &a, const V &b) { return md::mul(a, b); }
  __device__ static V mac(const V &c, const V &a, const V &b) { return md::add(c, md::mul(a, b)); }
  // b - a x, the update of the tail solve and the residual
  __device__ static V msub(const V &b, const V &a, const V &x) { return md::sub(b, md::mul(a, x)); }
  // the magnitude CPU_dbl_onenorm takes: |leading limb|
  __device__ static double mag(const V &a) { return fabs(R<K>::hi(a)); }
};
template <int K> struct NT<K, true> {
  typedef cplx<K> V;
  static constexpr int P = 2 * K;
  __device__ static V ld(const double *b, size_t m, size_t j) { return C<K>::load(b, m, j); }
  __device__ static void st(double *b, size_t m, size_t j, const V &v) { C<K>::store(b, m, j, v); }
  __device__ static V zero() { return C<K>::zero(); }
  __device__ static V one() { return C<K>::from(1.0, 0.0); }
  __device__ static V add(const V &a, const V &b) { return C<K>::add(a, b); }
  __device__ static V neg(const V &a) { return C<K>::neg(a); }
  // the first term and the inner loop of CPU_cmplx2_product
  __device__ static V mul(const V &a, const V &b) { return C<K>::mul(a, b); }
  __device__ static V mac(const V &c, const V &a, const V &b) {
    V z = c;
    C<K>::mac(z, a, b);
    return z;
  }
  // b - a x as CPU_cmplx2_qrbs_tail and CPU_cmplx2_linear_residue subtract
  // it: re -= a.re x.re, re += a.im x.im, im -= a.re x.im, im -= a.im x.re
  __device__ static V msub(const V &b, const V &a, const V &x) {
    V z;
    z.re = md::sub(b.re, md::mul(a.re, x.re));
    z.re = md::add(z.re, md::mul(a.im, x.im));
    z.im = md::sub(b.im, md::mul(a.re, x.im));
    z.im = md::sub(z.im, md::mul(a.im, x.re));
    return z;
  }
  // CPU_cmplx_onenorm's |re| + |im| of the leading limbs
  __device__ static double mag(const V &a) { return fabs(R<K>::hi(a.re)) + fabs(R<K>::hi(a.im)); }
};

// an LDS array of numbers, the P limbs of each side by side (K, or 2K when
// complex: a pair of limbs is one 16-byte access)
template <int K, bool CX = false> struct Arr {
  typedef typename NT<K, CX>::V T;
  static constexpr int P = NT<K, CX>::P;
  double *b;
  __device__ T ld(int j) const { return NT<K, CX>::ld(b + j * P, 1, 0); }
  __device__ void st(int j, const T &v) const { NT<K, CX>::st(b + j * P, 1, 0, v); }
  // the real (part 0) or imaginary (1) part of number j
  __device__ typename RealT<K>::type ldp(int j, int part) const {
    return R<K>::load(b + j * P + part * K, 1, 0);
  }
  __device__ void stp(int j, int part, const typename RealT<K>::type &v) const {
    R<K>::store(b + j * P + part * K, 1, 0, v);
  }
};

__device__ __forceinline__ bool all_zero(double a) { return a == 0.0; }
template <int K> __device__ __forceinline__ bool all_zero(const mdr<K> &a) {
  bool z = true;
#pragma unroll
  for (int i = 0; i < K; ++i) z = z && (a.x[i] == 0.0);
  return z;
}
__device__ __forceinline__ double limb(double a, int) { return a; }
template <int K> __device__ __forceinline__ double limb(const mdr<K> &a, int i) { return a.x[i]; }

// c ? a : b, limb by limb
__device__ __forceinline__ double choose(bool c, double a, double b) { return c ? a : b; }
template <int K> __device__ __forceinline__ mdr<K> choose(bool c, const mdr<K> &a, const mdr<K> &b) {
  mdr<K> r;
#pragma unroll
  for (int i = 0; i < K; ++i) r.x[i] = c ? a.x[i] : b.x[i];
  return r;
}

// carve an array of m numbers out of LDS
template <int K, bool CX = false> __device__ Arr<K, CX> carve(double *&p, int m) {
  Arr<K, CX> a{p};
  p += (size_t)NT<K, CX>::P * m;
  return a;
}

// largest |leading limb| of v[0..n-1], as CPU_dbl_onenorm computes it
// (Newton/dbl_onenorms_host.cpp:9-17): NaN when v[0] is NaN, later NaNs
// skipped.  Uniform over the team (every wavefront takes all n); every lane
// must call it.
template <int K, bool CX = false, class A = Arr<K, CX>>
__device__ double maxnorm(const A &v, int off, int n) {
  const int l = lane_id();
  double r = 0.0, v0 = 0.0;
  for (int i = l; i < n; i += 64) {
    const double a = NT<K, CX>::mag(v.ld(off + i));
    if (!(a <= r)) r = (a != a) ? r : a;
  }
  if (l == 0) v0 = NT<K, CX>::mag(v.ld(off));
  r = wave_fmax(r);
  v0 = __shfl(v0, 0, 64);
  return (v0 != v0) ? v0 : r;
}

// ------------------------------------------------ Householder QR (square)

// per-wave work arrays of the linear algebra; sc[0] = beta, sc[1] = v0, sc[2]
// = 1 when sigma = 0 (complex: sc[0] = beta and that flag, sc[1] = 1/v0)
template <int K, bool CX = false> struct LinWork {
  Arr<K, CX> q, r, v, w1, w2, wrk, sc;
};

// Q R = A for the n x n matrix given by the accessor a(r, c)
// (CPU_dbl2_factors_houseqr with CPU_dbl2_factors_house, leftRupdate and
// rightQupdate, Matrices/dbl2_factorizations.cpp:374-440, 534-566, 629-660)
template <int K, int TW, class A> __device__ void houseqr(int n, const A &a, const LinWork<K> &w) {
  typedef typename RealT<K>::type T;
  const int l = Team<TW>::id();
  for (int t = l; t < n * n; t += Team<TW>::N) {
    const int i = t / n, j = t % n;
    w.q.st(t, R<K>::from(i == j ? 1.0 : 0.0));
    w.r.st(t, a(i, j));
  }
  Team<TW>::sync();
  for (int k = 0; k < n; ++k) {
    const int m = n - k;
    // Householder vector of x = R[k..n-1][k]: sigma, mu, v0, beta in lane 0
    if (l == 0) {
      T sigma = R<K>::zero();
      for (int i = 1; i < m; ++i) sigma = add(sigma, sqr(w.r.ld((k + i) * n + k)));
      const bool zero = all_zero(sigma);
      w.sc.st(2, R<K>::from(zero ? 1.0 : 0.0));
      if (zero) {
        w.sc.st(0, R<K>::zero());
        w.sc.st(1, R<K>::from(1.0));
      } else {
        const T x0 = w.r.ld(k * n + k);
        T acc = sqr(x0);
        acc = add(acc, sigma);
        const T mu = R<K>::sqrt(acc);
        T v0;
        if (R<K>::hi(x0) <= 0.0) {
          v0 = sub(x0, mu);
        } else {
          acc = add(x0, mu);
          v0 = neg(div(sigma, acc));
        }
        const T v0p2 = sqr(v0);
        acc = add(sigma, v0p2);
        T beta = div(v0p2, acc);
        beta = mul_d(beta, 2.0);
        w.sc.st(0, beta);
        w.sc.st(1, v0);
      }
    }
    Team<TW>::sync();
    {
      const T v0 = w.sc.ld(1);
      const bool szero = R<K>::hi(w.sc.ld(2)) != 0.0;
      // v[i] = x[i] / v0 (x[i] unchanged when sigma = 0), v[0] = 1
      for (int i = l; i < m; i += Team<TW>::N) {
        if (i == 0) w.v.st(0, R<K>::from(1.0));
        else {
          const T xi = w.r.ld((k + i) * n + k);
          w.v.st(i, szero ? xi : div(xi, v0));
        }
      }
    }
    Team<TW>::sync();
    const T beta = w.sc.ld(0);
    // w1[j-k] = beta * sum_i R[i][j] v[i-k]
    for (int j = k + l; j < n; j += Team<TW>::N) {
      T s = R<K>::zero();
      for (int i = k; i < n; ++i) s = add(s, mul(w.r.ld(i * n + j), w.v.ld(i - k)));
      w.w1.st(j - k, mul(beta, s));
    }
    // w2[i] = beta * sum_{j>=k} Q[i][j] v[j-k]
    for (int i = l; i < n; i += Team<TW>::N) {
      T s = R<K>::zero();
      for (int j = k; j < n; ++j) s = add(s, mul(w.q.ld(i * n + j), w.v.ld(j - k)));
      w.w2.st(i, mul(beta, s));
    }
    Team<TW>::sync();
    // R[i][j] -= v[i-k] w1[j-k];  Q[i][j] -= w2[i] v[j-k]
    for (int t = l; t < m * m; t += Team<TW>::N) {
      const int i = k + t / m, j = k + t % m;
      w.r.st(i * n + j, sub(w.r.ld(i * n + j), mul(w.v.ld(i - k), w.w1.ld(j - k))));
    }
    for (int t = l; t < n * m; t += Team<TW>::N) {
      const int i = t / m, j = k + t % m;
      w.q.st(i * n + j, sub(w.q.ld(i * n + j), mul(w.w2.ld(i), w.v.ld(j - k))));
    }
    Team<TW>::sync();
  }
}

// x = R^{-1} Q^T b (CPU_dbl2_factors_qrbs and _backward): b = bv[bo..],
// x = xv[xo..]; b and x may be the same row.
template <int K, int TW, class BV>
__device__ void qrbs(int n, const LinWork<K> &w, const BV &bv, int bo, const Arr<K> &xv,
                     int xo) {
  typedef typename RealT<K>::type T;
  const int l = Team<TW>::id();
  for (int i = l; i < n; i += Team<TW>::N) {
    T s = R<K>::zero();
    for (int j = 0; j < n; ++j) s = add(s, mul(w.q.ld(j * n + i), bv.ld(bo + j)));
    w.wrk.st(i, s);
  }
  Team<TW>::sync();
  for (int i = l; i < n; i += Team<TW>::N) xv.st(xo + i, w.wrk.ld(i));
  Team<TW>::sync();
  // column sweep: row i receives the terms j = n-1 .. i+1 in that order
  for (int j = n - 1; j >= 0; --j) {
    if (l == j) xv.st(xo + j, div(xv.ld(xo + j), w.r.ld(j * n + j)));
    Team<TW>::sync();
    const T xj = xv.ld(xo + j);
    for (int i = l; i < j; i += Team<TW>::N) xv.st(xo + i, sub(xv.ld(xo + i), mul(w.r.ld(i * n + j), xj)));
    Team<TW>::sync();
  }
}

// The complex linear algebra works on components: two lanes form the real and
// the imaginary part of a number, each with the operations of the reference's
// host code in its order (a subtraction as the addition of the negated
// number, which gives the same limbs).  One lane per number took twice as
// long for each and the divisions of a row or a reflector one after another:
// 1.0 M cycles for a 6 x 6 quad-double factorization, 170 k for a solve.

// x - y or x + y
template <class T> __device__ __forceinline__ T add_or_sub(const T &x, const T &y, bool minus) {
  return add(x, choose(minus, neg(y), y));
}

// a value of lane src of the wavefront
__device__ __forceinline__ double from_lane(double a, int src) { return __shfl(a, src, 64); }
template <int K> __device__ __forceinline__ mdr<K> from_lane(const mdr<K> &a, int src) {
  mdr<K> r;
#pragma unroll
  for (int i = 0; i < K; ++i) r.x[i] = __shfl(a.x[i], src, 64);
  return r;
}

// Complex Q R = A (CPU_cmplx2_factors_houseqr with CPU_cmplx2_factors_house,
// leftRupdate and rightQupdate, Matrices/dbl2_factorizations.cpp:441-533,
// 567-627, 661-722, 766-822): the first wavefront forms the Householder
// vector's scalars (sigma = sum |x_i|^2, mu = sqrt(|x0|^2 + sigma) / |x0|, v0 =
// x0 - mu x0, beta = 2 |v0|^2 / (sigma + |v0|^2), 1/v0 = conj(v0) / |v0|^2),
// both roots in one call and the last three quotients in another, then the
// team v_i = x_i / v0, w1 = beta R^H v, w2 = beta Q v and the rank-one updates
// R -= v w1^H, Q -= w2 v^H, every entry in the reference's order.
template <int K, int TW, class A> __device__ void cx_houseqr(int n, const A &a, const LinWork<K, true> &w) {
  typedef typename RealT<K>::type T;
  typedef cplx<K> Z;
  const int l = Team<TW>::id(), N = Team<TW>::N;
  for (int t = l; t < n * n; t += N) {
    const int i = t / n, j = t % n;
    w.q.st(t, C<K>::from(i == j ? 1.0 : 0.0, 0.0));
    w.r.st(t, a(i, j));
  }
  Team<TW>::sync();
  for (int k = 0; k < n; ++k) {
    const int m = n - k;
    // the squares of the column's parts (w2 is free here)
    for (int t = l; t < 2 * m; t += N) w.w2.stp(t >> 1, t & 1, sqr(w.r.ldp((k + (t >> 1)) * n + k, t & 1)));
    Team<TW>::sync();
    if (l < 64) {
      T sigma = R<K>::zero();
      for (int i = 1; i < m; ++i) {
        sigma = add(sigma, w.w2.ldp(i, 0));
        sigma = add(sigma, w.w2.ldp(i, 1));
      }
      const bool zero = all_zero(sigma), odd = l & 1;
      T beta = R<K>::zero();
      Z inv = C<K>::from(1.0, 0.0);
      if (!zero) {
        const T xc = w.r.ldp(k * n + k, odd);
        const T sqrx0 = add(w.w2.ldp(0, 0), w.w2.ldp(0, 1));
        // even lanes: sqrt(|x0|^2 + sigma), odd lanes: |x0|
        const T rt = R<K>::sqrt(choose(odd, sqrx0, add(sqrx0, sigma)));
        T mu = from_lane(rt, 0);
        const T x0rad = from_lane(rt, 1);
        // even lanes: v0.re, odd lanes: v0.im
        T vc;
        if (all_zero(x0rad)) {
          vc = choose(odd, R<K>::zero(), neg(mu));
        } else {
          mu = div(mu, x0rad);
          vc = sub(xc, mul(mu, xc));
        }
        const T v2 = sqr(vc);
        const T sqrv0 = add(from_lane(v2, 0), from_lane(v2, 1));
        sigma = add(sigma, sqrv0);
        // lanes 0, 1: v0 / |v0|^2, lane 2: beta / 2
        const T qt = div(choose(l == 2, sqrv0, vc), choose(l == 2, sigma, sqrv0));
        beta = mul_d(from_lane(qt, 2), 2.0);
        inv.re = from_lane(qt, 0);
        inv.im = neg(from_lane(qt, 1));
      }
      if (l == 0) {
        Z z;
        z.re = beta;
        z.im = R<K>::from(zero ? 1.0 : 0.0);
        w.sc.st(0, z);
        w.sc.st(1, inv);
      }
    }
    Team<TW>::sync();
    const T beta = w.sc.ldp(0, 0);
    {
      const Z inv = w.sc.ld(1);
      const bool szero = R<K>::hi(w.sc.ldp(0, 1)) != 0.0;
      for (int t = l; t < 2 * m; t += N) {
        const int i = t >> 1, part = t & 1;
        if (i == 0) {
          w.v.stp(0, part, R<K>::from(part ? 0.0 : 1.0));
        } else {
          const Z x = w.r.ld((k + i) * n + k);
          T v = part ? x.im : x.re;
          if (!szero) v = add_or_sub(mul(v, inv.re), mul(part ? x.re : x.im, inv.im), part == 0);
          w.v.stp(i, part, v);
        }
      }
    }
    Team<TW>::sync();
    // w1[j-k] = beta * sum_i conj(R[i][j]) v[i-k], w2[i] = beta * sum_{j>=k}
    // Q[i][j] v[j-k]
    for (int t = l; t < 2 * (m + n); t += N) {
      const bool one = t < 2 * m;
      const int e = one ? t >> 1 : (t - 2 * m) >> 1, part = t & 1;
      T s = R<K>::zero();
      for (int q = 0; q < m; ++q) {
        const Z x = one ? w.r.ld((k + q) * n + k + e) : w.q.ld(e * n + k + q), v = w.v.ld(q);
        // w1: x.re v.re + x.im v.im, x.re v.im - x.im v.re
        // w2: x.re v.re - x.im v.im, x.im v.re + x.re v.im
        const bool im = part == 1, swap = !one && im;
        const T p1 = mul(swap ? x.im : x.re, (im && one) ? v.im : v.re);
        const T p2 = mul(swap ? x.re : x.im, (im && one) ? v.re : v.im);
        s = add(s, add_or_sub(p1, p2, one == im));
      }
      s = mul(beta, s);
      if (one) w.w1.stp(e, part, s);
      else w.w2.stp(e, part, s);
    }
    Team<TW>::sync();
    // R[i][j] -= v[i-k] conj(w1[j-k]);  Q[i][j] -= w2[i] conj(v[j-k])
    for (int t = l; t < 2 * (m + n) * m; t += N) {
      const int e = t >> 1, part = t & 1;
      const bool one = e < m * m;
      const int i = one ? e / m : (e - m * m) / m, j = one ? e % m : (e - m * m) % m;
      const Z x = one ? w.v.ld(i) : w.w2.ld(i), y = one ? w.w1.ld(j) : w.v.ld(j);
      const T z = add_or_sub(mul(part ? x.im : x.re, y.re), mul(part ? x.re : x.im, y.im), part == 1);
      const Arr<K, true> &M = one ? w.r : w.q;
      const int o = (one ? k + i : i) * n + k + j;
      M.stp(o, part, sub(M.ldp(o, part), z));
    }
    Team<TW>::sync();
  }
}

// x = R^{-1} Q^H b (CPU_cmplx2_factors_qrbs and _backward, Matrices/
// dbl2_factorizations.cpp:842-879, 142-200): b = bv[bo..], x = xv[xo..]; the
// reciprocals of R's diagonal, which the reference forms row by row, first
template <int K, int TW, class BV>
__device__ void cx_qrbs(int n, const LinWork<K, true> &w, const BV &bv, int bo,
                        const Arr<K, true> &xv, int xo) {
  typedef typename RealT<K>::type T;
  typedef cplx<K> Z;
  const int l = Team<TW>::id(), N = Team<TW>::N;
  for (int t = l; t < 2 * n; t += N) {
    const int i = t >> 1, part = t & 1;
    const Z u = w.r.ld(i * n + i);
    const T den = add(mul(u.re, u.re), mul(u.im, u.im));
    const T rc = div(part ? u.im : u.re, den);
    w.w1.stp(i, part, choose(part == 1, neg(rc), rc));
    T s = R<K>::zero();
    for (int j = 0; j < n; ++j) {
      // re: + q.re b.re + q.im b.im, im: + q.re b.im - q.im b.re
      const Z q = w.q.ld(j * n + i), b = bv.ld(bo + j);
      s = add(s, mul(q.re, part ? b.im : b.re));
      s = add_or_sub(s, mul(q.im, part ? b.re : b.im), part == 1);
    }
    w.wrk.stp(i, part, s);
  }
  Team<TW>::sync();
  for (int i = l; i < n; i += N) xv.st(xo + i, w.wrk.ld(i));
  Team<TW>::sync();
  for (int j = n - 1; j >= 0; --j) {
    T y;
    if (l < 2) {
      const Z x = xv.ld(xo + j), u = w.w1.ld(j);
      y = add_or_sub(mul(l ? x.im : x.re, u.re), mul(l ? x.re : x.im, u.im), l == 0);
    }
    Team<TW>::sync();
    if (l < 2) xv.stp(xo + j, l, y);
    Team<TW>::sync();
    const Z xj = xv.ld(xo + j);
    for (int t = l; t < 2 * j; t += N) {
      // re: - u.re x.re + u.im x.im, im: - u.im x.re - u.re x.im
      const int i = t >> 1, part = t & 1;
      const Z u = w.r.ld(i * n + j);
      T v = xv.ldp(xo + i, part);
      v = sub(v, mul(part ? u.im : u.re, xj.re));
      v = add_or_sub(v, mul(part ? u.re : u.im, xj.im), part == 1);
      xv.stp(xo + i, part, v);
    }
    Team<TW>::sync();
  }
}

// the real or complex factorization and solve
template <int K, bool CX, int TW, class A>
__device__ void any_houseqr(int n, const A &a, const LinWork<K, CX> &w) {
  if constexpr (CX) cx_houseqr<K, TW>(n, a, w);
  else houseqr<K, TW>(n, a, w);
}
template <int K, bool CX, int TW, class BV>
__device__ void any_qrbs(int n, const LinWork<K, CX> &w, const BV &bv, int bo, const Arr<K, CX> &xv, int xo) {
  if constexpr (CX) cx_qrbs<K, TW>(n, w, bv, bo, xv, xo);
  else qrbs<K, TW>(n, w, bv, bo, xv, xo);
}

struct Flags {
  int zeroQ, noqr, up, bs, newtail;
};

// lower block-triangular Toeplitz solve sum_{j<=k} A_j x_{k-j} = b_k
// (CPU_dbl2_qrbs_solve with _head and _tail); mat(j, r, c) = A_j[r][c];
// rhs and sol rows k at offsets k*n.  Uniform control flow.
template <int K, bool CX, int TW, class M, class BV>
__device__ void qrbs_solve(int n, int degp1, int tailidx, const M &mat, const BV &rhs,
                           const Arr<K, CX> &sol, const LinWork<K, CX> &w, Flags &f) {
  typedef typename NT<K, CX>::V T;
  const int l = Team<TW>::id();
  const double thr = threshold<K>();
  if (!(f.noqr && !f.zeroQ)) {
    const double nrm = maxnorm<K, CX>(rhs, 0, n);
    const bool small = (K == 1) ? (nrm + 1.0 == 1.0) : (nrm < thr);
    if (small) f.noqr = f.zeroQ ? 0 : 1;
    if (!f.noqr) {
      any_houseqr<K, CX, TW>(n, [&](int r, int c) { return mat(0, r, c); }, w);
      f.zeroQ = 0;
      any_qrbs<K, CX, TW>(n, w, rhs, 0, sol, 0);
    }
  }
  if (degp1 > 1) {
    int skipup = 0, skipbs = 0;
    bool firstbs = true;
    f.newtail = degp1;
    for (int i = tailidx; i < degp1; ++i) {
      if (maxnorm<K, CX>(sol, (i - 1) * n, n) < thr) {
        ++skipup;
      } else {
        const int npair = (degp1 - i) * n;
        // a component of an entry per lane
        constexpr int NC = CX ? 2 : 1;
        for (int t = l; t < NC * npair; t += Team<TW>::N) {
          const int e = t / NC, part = t % NC, j = i + e / n, k = e % n;
          typename RealT<K>::type b = rhs.ldp(j * n + k, part);
          for (int L = 0; L < n; ++L) {
            const T a = mat(j - i + 1, k, L), x = sol.ld((i - 1) * n + L);
            if constexpr (CX) {
              // as NT::msub: re -= a.re x.re, += a.im x.im; im -= a.re x.im, -= a.im x.re
              b = md::sub(b, md::mul(a.re, part ? x.im : x.re));
              b = add_or_sub(b, md::mul(a.im, part ? x.re : x.im), part == 1);
            } else {
              b = md::sub(b, md::mul(a, x));
            }
          }
          rhs.stp(j * n + k, part, b);
        }
      }
      Team<TW>::sync();
      const double nrm = maxnorm<K, CX>(rhs, i * n, n);
      if (nrm < thr || nrm > 1.0e+99) {
        ++skipbs;
        for (int j = l; j < n; j += Team<TW>::N) sol.st(i * n + j, NT<K, CX>::zero());
        Team<TW>::sync();
      } else {
        if (firstbs) {
          f.newtail = i;
          firstbs = false;
        }
        any_qrbs<K, CX, TW>(n, w, rhs, i * n, sol, i * n);
      }
    }
    f.up = skipup;
    f.bs = skipbs;
  }
}

// ---------------------------------------------- polynomial system values

// a monomial in one load: variable j in byte j of ix and its exponent in byte
// j of ex (the first eight), the number of variables, its coefficient series
struct MonoDesc {
  unsigned long long ix, ex;
  int nv, cm;
};

// the supports of a row system (shared by every system of a batch)
struct RowSys {
  int dim, nmono, nvmax, nbrmax, nfacmax;  // nfacmax: most factors of a common factor
  const int *monoptr, *nvr, *idxptr, *idx;
  const MonoDesc *desc;
  const int *exp;  // exponents parallel to idx, nullptr when all are 1
  // A system in the column representation (the column Newton method),
  // equation j holding monomial j of every column in column order: each
  // monomial is evaluated as CPU_dbl2_evaldiff does (a two-variable
  // monomial's value as (x_a x_b) c), the coefficient of row monomial m is
  // coefficient series desc[m].cm of the caller's ncff per system (unit series
  // when the coefficients are null: a monomial system), the constant is -1
  // in the last equation when negone and 0 elsewhere, and the right-hand
  // side of the linearized system is -(f - mb).
  int column, negone, ncff;
  // a monomial system (one monomial per equation): its value and
  // derivatives are stored, not added to zero, as
  // dbl2_linearize_evaldiff_output copies them (Newton/dbl2_systems_host.cpp:
  // 455-459, 506-513); an addition to zero renormalizes a quad double
  int assign;
};

// v * e, the derivative of a monomial times its exponent, with the
// multiplication by a double of each precision (ddf_mul_d_dd and its twins,
// as CPU_dbl2_evaluate_monomials does, Newton/dbl2_systems_host.cpp:103-110)
__device__ __forceinline__ double times_exp(double v, double e) { return e * v; }
template <int K> __device__ __forceinline__ mdr<K> times_exp(const mdr<K> &v, double e) {
  return mul_d(v, e);
}

// Two truncated products of series at once by the Dp lanes (lane k < Dw) of a
// component of a slot: coefficient k of x1*y1, then coefficient Dw-1-k of x2*y2,
// Dw + 1 multiply-adds on every lane where one lane per coefficient
// of one product leaves half of them idle (no second product: x2 = y2 = 0).  x1, ...: the rows' offsets in the
// array E; part: the component of a complex number this lane forms (0
// the real, 1 the imaginary part).  Each coefficient x_0 y_k, then += x_i
// y_{k-i}, in the order of CPU_dbl2_product and CPU_cmplx2_product
// (Convolutions/dbl2_convolutions_host.cpp:7-88).
template <int K, bool CX>
__device__ __forceinline__ void cprod2(const Arr<K, CX> &E, int part, int x1, int y1, int x2, int y2, int Dw,
                                       int k, typename RealT<K>::type &r1,
                                       typename RealT<K>::type &r2) {
  typedef typename RealT<K>::type T;
  // Issue of instructions bounds it (reading ahead made it slower), so the
  // trip count is uniform (without a second product the lanes go on with
  // numbers that nobody reads), the turn to the second product is selects on
  // one comparison, and up to double-double a sum starts from zero, to which
  // the first product is added without a rounding: 60 -> 49 instructions a
  // double-double multiply-add.
  constexpr int P = Arr<K, CX>::P;
  const double *px = E.b + x1 * P, *py = E.b + (y1 + k) * P, *const px2 = E.b + x2 * P,
               *const py2 = E.b + (y2 + Dw - 1 - k) * P;
  T acc = R<K>::zero(), first_sum = R<K>::zero();
  bool first = true;
#pragma unroll 2
  for (int it = 0; it <= Dw; ++it) {
    const T p = mul(R<K>::load(px + (CX && part ? K : 0), 1, 0), R<K>::load(py, 1, 0));
    acc = K <= 2 ? add(acc, p) : choose(first, p, add(acc, p));
    if constexpr (CX) {
      // re: xr yr - xi yi, im: xi yr + xr yi
      T q = mul(R<K>::load(px + (part ? 0 : K), 1, 0), R<K>::load(py + K, 1, 0));
      q = choose(part == 0, neg(q), q);
      acc = add(q, acc);
    }
    const bool turn = it == k;
    first_sum = choose(turn, acc, first_sum);
    if constexpr (K <= 2) acc = choose(turn, R<K>::zero(), acc);
    first = turn;
    px = turn ? px2 : px + P;
    py = turn ? py2 : py - P;
  }
  r1 = first_sum;
  r2 = acc;
}

// value and gradient series of every polynomial at X (working degree Dw-1):
// out row (p*(dim+1)+j) = d p / d x_j, row (p*(dim+1)+dim) = p, as
// CPU_dbl2_poly_evaldiff with CPU_dbl2_poly_speel and CPU_dbl2_speel
// (Polynomials/dbl2_polynomials_host.cpp, Convolutions/dbl2_monomials_host.cpp:28-87).
// A slot (Dp lanes per component) evaluates polynomials s, s + nslot, ...; its
// lane k of a component owns coefficients k and Dw-1-k of two products.
// cst/cff planes: cst + p*D, cff + m*D with plane strides.  E: the variables X
// at row offsets j*D, then the slots' work rows of length Dp: the coefficient
// C, the forward chain F (nvmax - 1 rows) and the backward chain B (nvmax - 2).
// A monomial's coefficient is staged in C; with exponents it is first
// multiplied by the common factor prod_j x_j^(e_j - 1), one factor at a time
// in the order of idx (the first loop of CPU_dbl2_evaluate_monomials,
// Newton/dbl2_systems_host.cpp:18-45), and each derivative contribution is
// multiplied by its exponent before it is added.  The chains advance together,
// one cprod2 a level; contributions to one row of OUT are added in the
// reference's order, the team in step (r1 before r2).
// (complex: the products of CPU_cmplx2_poly_evaldiff; no exponents)
template <int K, bool CX, int TW>
__device__ void eval_system(const RowSys &S, int D, int Dw, int Dp, const double *cst,
                            size_t cstride, const double *cff, size_t fstride,
                            const Arr<K, CX> &E, const Arr<K, CX> &OUT) {
  typedef typename RealT<K>::type T;
  typedef Team<TW> Tm;
  const int G = (CX ? 2 : 1) * Dp, nslot = Tm::N / G, s = Tm::id() / G, part = Tm::id() % G / Dp,
            k = Tm::id() % Dp;
  const int dim = S.dim, D1 = dim + 1, k2 = Dw - 1 - k;
  const int nv0 = S.nvmax > 0 ? S.nvmax : 1;
  const int rows = 1 + (nv0 - 1) + (nv0 > 2 ? nv0 - 2 : 0);
  const int C = dim * D + s * rows * Dp, F = C + Dp, B = F + (nv0 - 1) * Dp;
  auto keep = [&](int row, int q, const T &v) { E.stp(row + q, part, v); };
  // levels of the products of a monomial of nv variables, see below
  auto levels = [&](int nv) {
    return nv < 2 ? nv : nv == 2 ? 2 + (S.column != 0) : nv + (nv - 2) / 2;
  };
  int nlev = levels(S.nvmax);
  if (S.column && S.nvmax > 2 && nlev < 3) nlev = 3;
  for (int r0 = 0; r0 < dim; r0 += nslot) {
    const int p = r0 + s;
    const bool on = s < nslot && p < dim && k < Dw;
    if (on) {
      // column systems (cst null): 0, or -1 in the last equation
      T c0 = R<K>::zero();
      if (cst) c0 = R<K>::load(cst + (size_t)part * K * cstride, cstride, (size_t)p * D + k);
      else if (S.negone && p == dim - 1 && k == 0) c0 = R<K>::from(-1.0);
      OUT.stp((p * D1 + dim) * D + k, part, c0);
      for (int j = 0; j < dim; ++j) OUT.stp((p * D1 + j) * D + k, part, R<K>::zero());
    }
    const int m0 = on ? S.monoptr[p] : 0, nb = on ? S.monoptr[p + 1] - m0 : 0;
    // the next monomial's description and coefficient are loaded while the
    // current one is evaluated
    MonoDesc next{0, 0, 0, 0};
    T cnext = R<K>::zero();
    auto fetch = [&](int mi) {
      if (mi >= nb) return;
      next = S.desc[m0 + mi];
      cnext = R<K>::from(k == 0 ? 1.0 : 0.0);
      if (cff) cnext = R<K>::load(cff + (size_t)part * K * fstride, fstride, (size_t)next.cm * D + k);
    };
    fetch(0);
    for (int mi = 0; mi < S.nbrmax; ++mi) {
      const bool act = mi < nb;
      const MonoDesc md = next;
      const T c = cnext;
      fetch(mi + 1);
      const int mono = m0 + mi, nv = act ? md.nv : 0;
      const bool wide = nv > 8, powers = !CX && act && S.exp;
      auto var = [&](int j) { return wide ? S.idx[S.idxptr[mono] + j] : (int)(md.ix >> (8 * j)) & 255; };
      auto expo = [&](int j) { return wide ? S.exp[S.idxptr[mono] + j] : (int)(md.ex >> (8 * j)) & 255; };
      auto X = [&](int j) { return var(j) * D; };
      // v times the exponent of variable position j (positions with
      // exponent 1 are added as they are) to coefficient q of an OUT row
      auto addto = [&](int row, int q, const T &v, int j) {
        const int o = (p * D1 + row) * D + q;
        const int e = (powers && j >= 0) ? expo(j) : 1;
        const T ve = e > 1 ? times_exp(v, (double)e) : v;
        OUT.stp(o, part, (!CX && S.assign) ? ve : add(OUT.ldp(o, part), ve));
      };
      if (act) keep(C, k, c);
      Tm::sync();
      // the common factor, factor f of at most nfacmax: variable position fj
      // while e of its e_j - 1 factors are taken
      for (int f = 0, fj = 0, fe = 0; f < S.nfacmax; ++f) {
        T a = R<K>::zero(), unused;
        bool have = false;
        if (powers) {
          while (fj < nv && fe >= expo(fj) - 1) { ++fj; fe = 0; }
          have = fj < nv;
          if (have) {
            cprod2<K, CX>(E, part, X(fj), C, 0, 0, Dw, k, a, unused);
            ++fe;
          }
        }
        Tm::sync();
        if (have) keep(C, k, a);
        Tm::sync();
      }
      if (nv == 1) addto(var(0), k, E.ldp(C + k, part), 0);
      for (int t = 0; t < nlev; ++t) {
        // two products x1 y1, x2 y2 (-1: none), the rows that keep them (-1:
        // none), the OUT rows they are added to (-1: none) and the exponents'
        // positions: for nv > 2 the chains f_t = f_{t-1} x_t (f_{-1} = c) and
        // b_t = b_{t-1} x_{nv-2-t} (b_{-1} = x_{nv-1}) together, then c b_{nv-3}
        // beside f_{nv-2}, then the value f_{nv-1} and the cross products f_j
        // b_{nv-4-j} (the last f_{nv-3} x_{nv-1}) in order; for two variables
        // the value is (c x_a) x_b in a polynomial, (x_a x_b) c in a column
        // system
        int x1 = -1, y1 = 0, x2 = -1, y2 = 0, d1 = -1, d2 = -1, o1 = -1, o2 = -1, e1 = -1, e2 = -1;
        auto cross = [&](int j, int &x, int &y, int &o, int &e) {
          x = F + j * Dp;
          y = j < nv - 3 ? B + (nv - 4 - j) * Dp : X(nv - 1);
          o = var(j + 1);
          e = j + 1;
        };
        if (nv == 1) {
          if (t == 0) { x1 = X(0); y1 = C; o1 = dim; }
        } else if (nv == 2) {
          if (t == 0) {
            x1 = C; y1 = X(0); o1 = var(1); e1 = 1;
            if (!S.column) d1 = F;
            x2 = C; y2 = X(1); o2 = var(0); e2 = 0;
          } else if (!S.column) {
            if (t == 1) { x1 = F; y1 = X(1); o1 = dim; }
          } else if (t == 1) {
            x1 = X(0); y1 = X(1); d1 = F;
          } else if (t == 2) {
            x1 = F; y1 = C; o1 = dim;
          }
        } else if (nv > 2) {
          if (t <= nv - 3) {
            x1 = t ? F + (t - 1) * Dp : C; y1 = X(t); d1 = F + t * Dp;
            x2 = t ? B + (t - 1) * Dp : X(nv - 1); y2 = X(nv - 2 - t); d2 = B + t * Dp;
          } else if (t == nv - 2) {
            x1 = F + (t - 1) * Dp; y1 = X(t); d1 = F + t * Dp; o1 = var(nv - 1); e1 = nv - 1;
            x2 = B + (t - 1) * Dp; y2 = C; o2 = var(0); e2 = 0;
          } else if (t == nv - 1) {
            x1 = F + (t - 1) * Dp; y1 = X(t); o1 = dim;
            cross(0, x2, y2, o2, e2);
          } else {
            const int j = 2 * (t - nv) + 1;
            if (j <= nv - 3) cross(j, x1, y1, o1, e1);
            if (j + 1 <= nv - 3) cross(j + 1, x2, y2, o2, e2);
          }
        }
        T r1, r2;
        const bool have = act && x1 >= 0, two = have && x2 >= 0;
        if (have) {
          cprod2<K, CX>(E, part, x1, y1, two ? x2 : 0, two ? y2 : 0, Dw, k, r1, r2);
          if (o1 >= 0) addto(o1, k, r1, e1);
        }
        Tm::sync();
        if (have) {
          if (two && o2 >= 0) addto(o2, k2, r2, e2);
          if (d1 >= 0) keep(d1, k, r1);
          if (two && d2 >= 0) keep(d2, k2, r2);
        }
        Tm::sync();
      }
    }
  }
  Tm::sync();
}

// ------------------------------------------------------------ kernels

// numbers of a system's LDS: X with the evaluation's work rows behind it (E)
// and the solve's vectors and work arrays share it after X (SOLVE), the
// Jacobian and value series (OUT; the right-hand side is formed in place of
// the value rows), Q and R.
struct NewtonLayout {
  int E, X, SOLVE, OUT, Q;
  // P doubles per number: K (real) or 2K (complex)
  __host__ __device__ size_t bytes(int P) const {
    const int ev = E - X, tail = ev > SOLVE ? ev : SOLVE;
    return sizeof(double) * (size_t)P * ((size_t)X + tail + OUT + 2 * (size_t)Q);
  }
};

__host__ __device__ inline int pow2_at_least(int d) {
  int p = 1;
  while (p < d) p <<= 1;
  return p;
}

__host__ __device__ inline NewtonLayout newton_layout(const RowSys &S, int D, int TW, bool CX) {
  const int n = S.dim, nv = S.nvmax > 0 ? S.nvmax : 1, rows = 1 + (nv - 1) + (nv > 2 ? nv - 2 : 0);
  NewtonLayout L;
  L.X = n * D;
  // 64 TW lanes, one per coefficient (and component) of a slot's rows
  L.E = L.X + 64 * TW / (CX ? 2 : 1) * rows;
  L.SOLVE = D * n + 4 * n + 3;  // SOL, v, w1, w2, wrk, scalars
  L.OUT = n * (n + 1) * D;
  L.Q = n * n;
  return L;
}

// wavefronts of a team: one while the systems fill the chip; with fewer
// systems than 2 per compute unit (or more lanes than a wavefront's needed for
// one slot) as many as evaluate all polynomials at once, up to 4
inline int team_waves(const RowSys &S, int D, bool CX, int nsys) {
  const int G = (CX ? 2 : 1) * pow2_at_least(D);
  int tw = G > 64 ? 2 : 1;
  if (nsys <= 512)
    while (tw < 4 && 64 * tw < S.dim * G) tw *= 2;
  return tw;
}

template <int K, bool CX = false>
__device__ LinWork<K, CX> carve_lin(double *&p, int n) {
  LinWork<K, CX> w;
  w.q = carve<K, CX>(p, n * n); w.r = carve<K, CX>(p, n * n); w.v = carve<K, CX>(p, n);
  w.w1 = carve<K, CX>(p, n); w.w2 = carve<K, CX>(p, n); w.wrk = carve<K, CX>(p, n);
  w.sc = carve<K, CX>(p, 3);
  return w;
}

// x [K][nsys][dim][D] in/out; cst [K][nc][dim][D], cff [K][nf][ncff][D] with
// nc, nf = nsys or 1 (shared); logs [nsys][nbsteps]; hist
// [nbsteps][K][nsys][dim][D]; Q, R [K][nsys][dim][dim].  Column systems:
// cst null, cff null for unit coefficients, mb [K][nm][dim][D] (nm = nsys
// or 1); rows: mb null.
template <int K, bool CX, int TW>
__global__ void __launch_bounds__(64 * TW)
row_newton_kernel(RowSys S, int deg, int nbsteps, int nsys, const double *cst, int cshared,
                  const double *cff, int fshared, const double *mb, int mshared, double *x,
                  int *steps_out, int *wdeg_out, int *tail_out, int *up_out, int *bs_out,
                  double *hist, double *Qo, double *Ro) {
  typedef NT<K, CX> N;
  typedef Team<TW> Tm;
  extern __shared__ __align__(16) double lds[];
  const int D = deg + 1, n = S.dim, D1 = n + 1;
  const NewtonLayout L = newton_layout(S, D, TW, CX);
  const int l = Tm::id(), sysid = blockIdx.x;
  double *p = lds;
  const Arr<K, CX> OUT = carve<K, CX>(p, L.OUT);
  LinWork<K, CX> w;
  w.q = carve<K, CX>(p, L.Q);
  w.r = carve<K, CX>(p, L.Q);
  // X and the evaluation's work rows, whose place is the solve's arrays'
  // between evaluations
  const Arr<K, CX> E{p};
  auto sub_arr = [&](int off) { return Arr<K, CX>{E.b + (L.X + off) * N::P}; };
  const Arr<K, CX> SOL = sub_arr(0);
  w.v = sub_arr(D * n); w.w1 = sub_arr(D * n + n); w.w2 = sub_arr(D * n + 2 * n);
  w.wrk = sub_arr(D * n + 3 * n); w.sc = sub_arr(D * n + 4 * n);
  // right-hand side k of equation i in place of the value's coefficient
  struct Rhs {
    Arr<K, CX> a;
    int n, D;
    __device__ int at(int t) const { return (t % n * (n + 1) + n) * D + t / n; }
    __device__ typename N::V ld(int t) const { return a.ld(at(t)); }
    __device__ void st(int t, const typename N::V &v) const { a.st(at(t), v); }
    __device__ typename RealT<K>::type ldp(int t, int part) const { return a.ldp(at(t), part); }
    __device__ void stp(int t, int part, const typename RealT<K>::type &v) const { a.stp(at(t), part, v); }
  };
  const Rhs RHS{OUT, n, D};
  const size_t xs = (size_t)nsys * n * D, xb = (size_t)sysid * n * D;
  const size_t cs = (size_t)(cshared ? 1 : nsys) * n * D;
  const size_t fs = (size_t)(fshared ? 1 : nsys) * S.ncff * D;
  const size_t ms = (size_t)(mshared ? 1 : nsys) * n * D, mo = mshared ? 0 : (size_t)sysid * n * D;
  const double *cbase = cst ? cst + (cshared ? 0 : (size_t)sysid * n * D) : nullptr;
  const double *fbase = cff ? cff + (fshared ? 0 : (size_t)sysid * S.ncff * D) : nullptr;
  for (int t = l; t < n * D; t += Tm::N) E.st(t, N::ld(x, xs, xb + t));
  Tm::sync();
  auto jac = [&](int j, int r, int c) { return OUT.ld((r * D1 + c) * D + j); };
  Flags f{1, 0, 0, 0, 1};
  int tailidx = 1, wrkdeg = 0, stepcnt = 0;
  for (int step = 0; step < nbsteps; ++step) {
    const int Dw = wrkdeg + 1;
    eval_system<K, CX, TW>(S, D, Dw, pow2_at_least(Dw), cbase, cs, fbase, fs, E, OUT);
    for (int t = l; t < Dw * n; t += Tm::N) {
      const int kk = t / n, i = t % n;
      const typename N::V fv = RHS.ld(t);
      if constexpr (CX) {
        RHS.st(t, N::neg(fv));
      } else {
        // -(f - mb) as dbl2_define_rhs (Newton/dbl2_systems_host.cpp:626-659)
        RHS.st(t, mb ? N::neg(md::sub(fv, N::ld(mb, ms, mo + (size_t)i * D + kk))) : N::neg(fv));
      }
      SOL.st(t, N::zero());
    }
    Tm::sync();
    f.newtail = tailidx;
    qrbs_solve<K, CX, TW>(n, Dw, tailidx, jac, RHS, SOL, w, f);
    tailidx = f.newtail;
    Tm::sync();
    for (int t = l; t < n * Dw; t += Tm::N) {
      const int i = t / Dw, kk = t % Dw;
      if (kk >= tailidx - 1) E.st(i * D + kk, N::add(E.ld(i * D + kk), SOL.ld(kk * n + i)));
    }
    Tm::sync();
    if (l == 0) {
      const size_t o = (size_t)sysid * nbsteps + step;
      if (wdeg_out) wdeg_out[o] = wrkdeg;
      if (tail_out) tail_out[o] = tailidx;
      if (up_out) up_out[o] = f.up;
      if (bs_out) bs_out[o] = f.bs;
    }
    if (hist) {
      double *h = hist + (size_t)step * N::P * xs;
      for (int t = l; t < n * D; t += Tm::N) N::st(h, xs, xb + t, E.ld(t));
    }
    ++stepcnt;
    if (tailidx >= deg) break;
    wrkdeg = wrkdeg + 1 + wrkdeg / 2;
    if (wrkdeg > deg) wrkdeg = deg;
  }
  for (int t = l; t < n * D; t += Tm::N) N::st(x, xs, xb + t, E.ld(t));
  const size_t qs = (size_t)nsys * n * n, qb = (size_t)sysid * n * n;
  for (int t = l; t < n * n; t += Tm::N) {
    if (Qo) N::st(Qo, qs, qb + t, w.q.ld(t));
    if (Ro) N::st(Ro, qs, qb + t, w.r.ld(t));
  }
  if (l == 0 && steps_out) steps_out[sysid] = stepcnt;
}

// batched Householder QR of n x n matrices A [K][nb][n][n] -> Q, R
template <int K, bool CX>
__global__ void __launch_bounds__(512)
houseqr_kernel(int n, int nb, const double *A, double *Qo, double *Ro) {
  typedef NT<K, CX> N;
  extern __shared__ __align__(16) double lds[];
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int b = blockIdx.x * (blockDim.x >> 6) + wave;
  if (b >= nb) return;
  const size_t per = (size_t)N::P * (2 * n * n + 4 * n + 3);
  double *p = lds + (size_t)wave * per;
  const LinWork<K, CX> w = carve_lin<K, CX>(p, n);
  const size_t s = (size_t)nb * n * n, o = (size_t)b * n * n;
  any_houseqr<K, CX, 1>(n, [&](int r, int c) { return N::ld(A, s, o + (size_t)r * n + c); }, w);
  for (int t = l; t < n * n; t += 64) {
    N::st(Qo, s, o + t, w.q.ld(t));
    N::st(Ro, s, o + t, w.r.ld(t));
  }
}

// batched Toeplitz solve: mat [K][nb][degp1][n][n], rhs/sol [K][nb][degp1][n]
// (in/out), Q/R [K][nb][n][n] (in/out), flags [nb][5] (zeroQ, noqr, up, bs,
// newtail; in/out)
template <int K, bool CX>
__global__ void __launch_bounds__(512)
qrbs_solve_kernel(int n, int degp1, int tailidx, int nb, const double *mat, double *rhs,
                  double *sol, double *Qio, double *Rio, int *flags) {
  typedef NT<K, CX> N;
  extern __shared__ __align__(16) double lds[];
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int b = blockIdx.x * (blockDim.x >> 6) + wave;
  if (b >= nb) return;
  const size_t per = (size_t)N::P * (2 * n * n + 4 * n + 3 + 2 * degp1 * n);
  double *p = lds + (size_t)wave * per;
  const LinWork<K, CX> w = carve_lin<K, CX>(p, n);
  const Arr<K, CX> RHS = carve<K, CX>(p, degp1 * n), SOL = carve<K, CX>(p, degp1 * n);
  const size_t vs = (size_t)nb * degp1 * n, vo = (size_t)b * degp1 * n;
  const size_t qs = (size_t)nb * n * n, qo = (size_t)b * n * n;
  const size_t ms = (size_t)nb * degp1 * n * n, mo = (size_t)b * degp1 * n * n;
  for (int t = l; t < degp1 * n; t += 64) {
    RHS.st(t, N::ld(rhs, vs, vo + t));
    SOL.st(t, N::ld(sol, vs, vo + t));
  }
  for (int t = l; t < n * n; t += 64) {
    w.q.st(t, N::ld(Qio, qs, qo + t));
    w.r.st(t, N::ld(Rio, qs, qo + t));
  }
  wsync();
  Flags f{flags[b * 5], flags[b * 5 + 1], flags[b * 5 + 2], flags[b * 5 + 3], flags[b * 5 + 4]};
  auto m = [&](int j, int r, int c) { return N::ld(mat, ms, mo + ((size_t)j * n + r) * n + c); };
  qrbs_solve<K, CX, 1>(n, degp1, tailidx, m, RHS, SOL, w, f);
  for (int t = l; t < degp1 * n; t += 64) {
    N::st(rhs, vs, vo + t, RHS.ld(t));
    N::st(sol, vs, vo + t, SOL.ld(t));
  }
  for (int t = l; t < n * n; t += 64) {
    N::st(Qio, qs, qo + t, w.q.ld(t));
    N::st(Rio, qs, qo + t, w.r.ld(t));
  }
  if (l == 0) {
    flags[b * 5] = f.zeroQ; flags[b * 5 + 1] = f.noqr; flags[b * 5 + 2] = f.up;
    flags[b * 5 + 3] = f.bs; flags[b * 5 + 4] = f.newtail;
  }
}

// r_i = b_i - sum_{j <= i-tailidx} A_j x_{i-j} for i >= tailidx
// (CPU_dbl2_linear_residue, Newton/dbl2_bals_host.cpp:548-600); one lane per
// residual entry; resmax [K][nb] = entry of largest |leading limb|, the first
// such entry in the reference's scan order.
template <int K, bool CX>
__global__ void __launch_bounds__(512)
linear_residue_kernel(int n, int degp1, int tailidx, int nb, const double *mat,
                      const double *rhs, const double *sol, double *res, double *resmax) {
  typedef NT<K, CX> N;
  typedef typename N::V T;
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int b = blockIdx.x * (blockDim.x >> 6) + wave;
  if (b >= nb) return;
  const size_t vs = (size_t)nb * degp1 * n, vo = (size_t)b * degp1 * n;
  const size_t ms = (size_t)nb * degp1 * n * n, mo = (size_t)b * degp1 * n * n;
  double best = 0.0;
  int bidx = -1;
  for (int t = tailidx * n + l; t < degp1 * n; t += 64) {
    const int i = t / n, L = t % n;
    T r = N::ld(rhs, vs, vo + t);
    for (int j = 0; j <= i - tailidx; ++j)
      for (int k = 0; k < n; ++k)
        r = N::msub(r, N::ld(mat, ms, mo + ((size_t)j * n + L) * n + k),
                    N::ld(sol, vs, vo + (size_t)(i - j) * n + k));
    N::st(res, vs, vo + t, r);
    const double a = N::mag(r);
    if (a > best) { best = a; bidx = t; }
  }
  // the scan keeps the first strictly larger entry: largest value, then the
  // smallest index among equal values
  for (int m = 1; m < 64; m <<= 1) {
    const double ob = __shfl_xor(best, m, 64);
    const int oi = __shfl_xor(bidx, m, 64);
    if (ob > best || (ob == best && oi >= 0 && (bidx < 0 || oi < bidx))) { best = ob; bidx = oi; }
  }
  if (l == 0) {
    T r = N::zero();
    if (bidx >= 0) r = N::ld(res, vs, vo + bidx);
#pragma unroll
    for (int i = 0; i < K; ++i) {
      // complex: |re| + |im| limb by limb, as CPU_cmplx2_linear_residue
      if constexpr (CX) resmax[(size_t)i * nb + b] = fabs(limb(r.re, i)) + fabs(limb(r.im, i));
      else resmax[(size_t)i * nb + b] = fabs(limb(r, i));
    }
  }
}

int waves_for(size_t per_wave, int *waves) {
  int dev = 0, ldsmax = 0;
  PHC_HIP(hipGetDevice(&dev));
  PHC_HIP(hipDeviceGetAttribute(&ldsmax, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  const size_t cap = (size_t)ldsmax < LDS_LIMIT ? (size_t)ldsmax : LDS_LIMIT;
  PHC_REQUIRE(per_wave <= cap, "problem too large for the LDS of one workgroup");
  int wv = (int)(cap / per_wave);
  if (wv > 8) wv = 8;
  *waves = wv;
  return 0;
}

}  // namespace

struct phc_rowsys {
  RowSys S;
  int *dmem;
  MonoDesc *ddesc;
  int nbrcol;  // column systems: the number of columns (0 for row systems)
};

namespace {
// the monomials' descriptions (cmap: coefficient series of each, null: its own)
int upload_desc(phc_rowsys *s, int nmono, const int *nvr, const int *idxptr, const int *idx,
                const int *exp, const int *cmap) {
  std::vector<MonoDesc> h(nmono > 0 ? nmono : 1, MonoDesc{0, 0, 0, 0});
  for (int m = 0; m < nmono; ++m) {
    h[m].nv = nvr[m];
    h[m].cm = cmap ? cmap[m] : m;
    for (int j = 0; j < nvr[m] && j < 8; ++j) {
      h[m].ix |= (unsigned long long)idx[idxptr[m] + j] << (8 * j);
      h[m].ex |= (unsigned long long)(exp ? exp[idxptr[m] + j] : 1) << (8 * j);
    }
  }
  if (!s->ddesc) PHC_HIP(hipMalloc(&s->ddesc, sizeof(MonoDesc) * h.size()));
  PHC_HIP(hipMemcpy(s->ddesc, h.data(), sizeof(MonoDesc) * h.size(), hipMemcpyHostToDevice));
  s->S.desc = s->ddesc;
  return 0;
}
}  // namespace

extern "C" {

int phc_rowsys_create_exp(phc_rowsys **out, int dim, const int *monoptr, const int *nvr,
                          const int *idxptr, const int *idx, const int *exp);
int phc_rowsys_destroy(phc_rowsys *s);

int phc_rowsys_create(phc_rowsys **out, int dim, const int *monoptr, const int *nvr,
                      const int *idxptr, const int *idx) {
  return phc_rowsys_create_exp(out, dim, monoptr, nvr, idxptr, idx, nullptr);
}

int phc_rowsys_create_exp(phc_rowsys **out, int dim, const int *monoptr, const int *nvr,
                          const int *idxptr, const int *idx, const int *exp) {
  PHC_REQUIRE(out && monoptr && nvr && idxptr, "phc_rowsys_create: null argument");
  PHC_REQUIRE(dim >= 1 && dim <= 64, "phc_rowsys_create: dim must be in 1..64");
  const int nmono = monoptr[dim];
  PHC_REQUIRE(monoptr[0] == 0 && nmono >= 0, "phc_rowsys_create: bad monomial pointers");
  int nvmax = 0, nbrmax = 0;
  for (int i = 0; i < dim; ++i) {
    PHC_REQUIRE(monoptr[i + 1] >= monoptr[i], "phc_rowsys_create: bad monomial pointers");
    if (monoptr[i + 1] - monoptr[i] > nbrmax) nbrmax = monoptr[i + 1] - monoptr[i];
  }
  PHC_REQUIRE(idxptr[0] == 0, "phc_rowsys_create: bad index pointers");
  for (int m = 0; m < nmono; ++m) {
    PHC_REQUIRE(nvr[m] >= 1 && nvr[m] <= dim && idxptr[m + 1] - idxptr[m] == nvr[m],
                "phc_rowsys_create: monomial variable counts and index pointers disagree");
    for (int j = idxptr[m]; j < idxptr[m + 1]; ++j)
      PHC_REQUIRE(idx && idx[j] >= 0 && idx[j] < dim, "phc_rowsys_create: variable index out of range");
    if (nvr[m] > nvmax) nvmax = nvr[m];
  }
  const int nidx = idxptr[nmono];
  bool any_exp = false;
  int nfacmax = 0;
  for (int j = 0; exp && j < nidx; ++j) {
    PHC_REQUIRE(exp[j] >= 1 && exp[j] <= 64, "phc_rowsys_create: exponents must be in 1..64");
    any_exp = any_exp || exp[j] > 1;
  }
  for (int m = 0; exp && m < nmono; ++m) {
    int nfac = 0;
    for (int j = idxptr[m]; j < idxptr[m + 1]; ++j) nfac += exp[j] - 1;
    if (nfac > nfacmax) nfacmax = nfac;
  }
  const size_t ints = (size_t)(dim + 1) + 2 * (size_t)nmono + 1 + nidx + (any_exp ? nidx : 0);
  phc_rowsys *s = new phc_rowsys();
  if (hipMalloc(&s->dmem, sizeof(int) * (ints > 0 ? ints : 1)) != hipSuccess) {
    delete s;
    phc::set_error("phc_rowsys_create: hipMalloc failed");
    return -1;
  }
  int *p = s->dmem;
  std::vector<int> h;
  h.insert(h.end(), monoptr, monoptr + dim + 1);
  h.insert(h.end(), nvr, nvr + nmono);
  h.insert(h.end(), idxptr, idxptr + nmono + 1);
  if (nidx > 0) h.insert(h.end(), idx, idx + nidx);
  if (any_exp) h.insert(h.end(), exp, exp + nidx);
  PHC_HIP(hipMemcpy(p, h.data(), sizeof(int) * h.size(), hipMemcpyHostToDevice));
  s->S.dim = dim; s->S.nmono = nmono; s->S.nvmax = nvmax; s->S.nbrmax = nbrmax;
  s->S.nfacmax = nfacmax;
  s->S.monoptr = p; s->S.nvr = p + dim + 1; s->S.idxptr = p + dim + 1 + nmono;
  s->S.idx = p + dim + 1 + 2 * nmono + 1;
  s->S.exp = any_exp ? s->S.idx + nidx : nullptr;
  s->S.ncff = nmono;
  if (upload_desc(s, nmono, nvr, idxptr, idx, exp, nullptr) != 0) {
    phc_rowsys_destroy(s);
    return -1;
  }
  *out = s;
  return 0;
}

int phc_colsys_create(phc_rowsys **out, int dim, int nbrcol, const int *nvr, const int *idx,
                      const int *exps) {
  PHC_REQUIRE(out && nvr, "phc_colsys_create: null argument");
  PHC_REQUIRE(dim >= 1 && dim <= 64, "phc_colsys_create: dim must be in 1..64");
  PHC_REQUIRE(nbrcol >= 1 && nbrcol <= 64, "phc_colsys_create: nbrcol must be in 1..64");
  PHC_REQUIRE(nbrcol == 1 || exps == nullptr,
              "phc_colsys_create: exponents are for monomial systems (nbrcol = 1) only");
  const int ncff = nbrcol * dim;
  std::vector<int> iptr(ncff + 1, 0);
  for (int m = 0; m < ncff; ++m) {
    PHC_REQUIRE(nvr[m] >= (nbrcol == 1 ? 1 : 0) && nvr[m] <= dim,
                "phc_colsys_create: monomial variable count out of range");
    iptr[m + 1] = iptr[m] + nvr[m];
  }
  // equation j: monomial j of every column in column order (the order in
  // which CPU_dbl2_evaluate_columns adds them, Newton/dbl2_systems_host.cpp:
  // 291-323), empty monomials left out
  std::vector<int> monoptr(dim + 1, 0), rnvr, ridxptr(1, 0), ridx, rexp, cmap;
  for (int j = 0; j < dim; ++j) {
    for (int c = 0; c < nbrcol; ++c) {
      const int m = c * dim + j;
      if (nvr[m] == 0) continue;
      rnvr.push_back(nvr[m]);
      cmap.push_back(m);
      for (int k = iptr[m]; k < iptr[m + 1]; ++k) {
        PHC_REQUIRE(idx, "phc_colsys_create: null index array");
        ridx.push_back(idx[k]);
        if (exps) rexp.push_back(exps[k]);
      }
      ridxptr.push_back((int)ridx.size());
    }
    monoptr[j + 1] = (int)rnvr.size();
  }
  for (size_t m = 0; m < rnvr.size(); ++m)
    for (int a = ridxptr[m]; a < ridxptr[m + 1]; ++a)
      for (int b = a + 1; b < ridxptr[m + 1]; ++b)
        PHC_REQUIRE(ridx[a] != ridx[b], "phc_colsys_create: repeated variable in a monomial");
  phc_rowsys *s = nullptr;
  const int rc = phc_rowsys_create_exp(&s, dim, monoptr.data(), rnvr.data(), ridxptr.data(),
                                       ridx.data(), exps ? rexp.data() : nullptr);
  if (rc != 0) return rc;
  s->nbrcol = nbrcol;
  s->S.column = 1;
  s->S.negone = nbrcol > 1;
  s->S.assign = nbrcol == 1;
  s->S.ncff = ncff;
  if (upload_desc(s, (int)rnvr.size(), rnvr.data(), ridxptr.data(), ridx.data(),
                  exps ? rexp.data() : nullptr, cmap.data()) != 0) {
    phc_rowsys_destroy(s);
    return -1;
  }
  *out = s;
  return 0;
}

int phc_rowsys_destroy(phc_rowsys *s) {
  if (!s) return 0;
  hipError_t e = hipFree(s->dmem);
  if (s->ddesc) {
    const hipError_t e1 = hipFree(s->ddesc);
    if (e == hipSuccess) e = e1;
  }
  delete s;
  if (e != hipSuccess) {
    phc::set_error("phc_rowsys_destroy: hipFree failed");
    return -1;
  }
  return 0;
}

int phc_rowsys_lds_bytes(const phc_rowsys *s, int K, int deg, size_t *bytes) {
  PHC_REQUIRE(s && bytes, "phc_rowsys_lds_bytes: null argument");
  PHC_REQUIRE(deg >= 0 && deg <= 63, "phc_rowsys_lds_bytes: deg must be in 0..63");
  *bytes = newton_layout(s->S, deg + 1, 1, false).bytes(K);
  return 0;
}

}  // extern "C"

namespace {

// the staggered row Newton, real (P = K planes) or complex (2K)
template <bool CX>
int row_newton(phc_rowsys *s, int K, int deg, int nbsteps, int nsys, const double *cst,
               int cst_shared, const double *cff, int cff_shared, const double *mb,
               int mb_shared, double *x, int *steps, int *wdeg, int *tail, int *up, int *bs,
               double *history, double *Q, double *R, void *stream, const char *fn) {
  PHC_REQUIRE(s, std::string(fn) + ": null system");
  const bool column = s->S.column != 0;
  PHC_REQUIRE(!column || mb, std::string(fn) + ": a column system goes to phc_column_newton "
                                               "with its right-hand side");
  if (CX) {
    PHC_REQUIRE(K == 2 || K == 4, std::string(fn) + ": K must be 2 or 4");
    PHC_REQUIRE(s->S.exp == nullptr, std::string(fn) + ": exponents above 1 are real only");
  } else {
    PHC_REQUIRE(K == 1 || K == 2 || K == 4, std::string(fn) + ": K must be 1, 2 or 4");
  }
  PHC_REQUIRE(deg >= 0 && deg <= 63, std::string(fn) + ": deg must be in 0..63");
  PHC_REQUIRE(nbsteps >= 0 && nsys >= 0, std::string(fn) + ": negative size");
  if (column) {
    PHC_REQUIRE(!CX, std::string(fn) + ": column systems are real");
    PHC_REQUIRE(x && (cff || s->nbrcol == 1),
                std::string(fn) + ": null coefficient or series array");
  } else {
    PHC_REQUIRE(cst && cff && x, std::string(fn) + ": null coefficient or series array");
  }
  if (nsys == 0 || nbsteps == 0) return 0;
  const int P = CX ? 2 * K : K;
  int tw = team_waves(s->S, deg + 1, CX, nsys);
  // more wavefronts take more work rows
  while (tw > 1 && newton_layout(s->S, deg + 1, tw, CX).bytes(P) > LDS_LIMIT && 32 * tw >= (CX ? 2 : 1) * pow2_at_least(deg + 1)) tw /= 2;
  const size_t lds = newton_layout(s->S, deg + 1, tw, CX).bytes(P);
  int wv = 0;
  if (waves_for(lds, &wv) != 0) return -2;
  hipStream_t st = (hipStream_t)stream;
#define LAUNCH_TEAM(KK, TW)                                                                   \
  do {                                                                                        \
    PHC_HIP(hipFuncSetAttribute((const void *)row_newton_kernel<KK, CX, TW>,                 \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));       \
    hipLaunchKernelGGL((row_newton_kernel<KK, CX, TW>), dim3(nsys), dim3(64 * TW), lds, st,   \
                       s->S, deg, nbsteps, nsys, cst, cst_shared, cff, cff_shared, mb,        \
                       mb_shared, x, steps, wdeg, tail, up, bs, history, Q, R);               \
  } while (0)
#define LAUNCH(KK)                                                                            \
  do {                                                                                        \
    if (tw == 1) LAUNCH_TEAM(KK, 1);                                                          \
    else if (tw == 2) LAUNCH_TEAM(KK, 2);                                                     \
    else LAUNCH_TEAM(KK, 4);                                                                  \
  } while (0)
  if (K == 1 && !CX) LAUNCH(1);
  else if (K == 2) LAUNCH(2);
  else LAUNCH(4);
#undef LAUNCH_TEAM
#undef LAUNCH
  PHC_HIP(hipGetLastError());
  return 0;
}

template <bool CX>
int houseqr_batch(int K, int n, int nbatch, const double *A, double *Q, double *R, void *stream,
                  const char *fn) {
  // complex octo-double (K = 8) is refused: its first device run stalled
  // (a launch of houseqr_kernel<8, true> that did not return), cause not
  // established
  PHC_REQUIRE(CX ? (K == 2 || K == 4) : (K == 1 || K == 2 || K == 4),
              std::string(fn) + (CX ? ": K must be 2 or 4" : ": K must be 1, 2 or 4"));
  PHC_REQUIRE(n >= 1 && n <= 64 && nbatch >= 0, std::string(fn) + ": n must be in 1..64");
  PHC_REQUIRE(A && Q && R, std::string(fn) + ": null array");
  if (nbatch == 0) return 0;
  const size_t per = sizeof(double) * (CX ? 2 * K : K) * (2 * (size_t)n * n + 4 * n + 3);
  int wv = 0;
  if (waves_for(per, &wv) != 0) return -2;
  const int grid = (nbatch + wv - 1) / wv;
  hipStream_t st = (hipStream_t)stream;
#define LAUNCH(KK)                                                                            \
  do {                                                                                        \
    PHC_HIP(hipFuncSetAttribute((const void *)houseqr_kernel<KK, CX>,                        \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)(per * wv))); \
    hipLaunchKernelGGL((houseqr_kernel<KK, CX>), dim3(grid), dim3(64 * wv), per * wv, st, n,  \
                       nbatch, A, Q, R);                                                      \
  } while (0)
  if (K == 1 && !CX) LAUNCH(1);
  else if (K == 2) LAUNCH(2);
  else LAUNCH(4);
#undef LAUNCH
  PHC_HIP(hipGetLastError());
  return 0;
}

template <bool CX>
int qrbs_solve_batch(int K, int n, int degp1, int tailidx, int nbatch, const double *mat,
                     double *rhs, double *sol, double *Q, double *R, int *flags, void *stream,
                     const char *fn) {
  // complex octo-double (K = 8) is refused: its first device run stalled
  // (a launch of houseqr_kernel<8, true> that did not return), cause not
  // established
  PHC_REQUIRE(CX ? (K == 2 || K == 4) : (K == 1 || K == 2 || K == 4),
              std::string(fn) + (CX ? ": K must be 2 or 4" : ": K must be 1, 2 or 4"));
  PHC_REQUIRE(n >= 1 && n <= 64 && degp1 >= 1 && degp1 <= 64 && nbatch >= 0,
              std::string(fn) + ": n and degp1 must be in 1..64");
  PHC_REQUIRE(tailidx >= 1, std::string(fn) + ": tailidx must be at least 1");
  PHC_REQUIRE(mat && rhs && sol && Q && R && flags, std::string(fn) + ": null array");
  if (nbatch == 0) return 0;
  const size_t per =
      sizeof(double) * (CX ? 2 * K : K) * (2 * (size_t)n * n + 4 * n + 3 + 2 * (size_t)degp1 * n);
  int wv = 0;
  if (waves_for(per, &wv) != 0) return -2;
  const int grid = (nbatch + wv - 1) / wv;
  hipStream_t st = (hipStream_t)stream;
#define LAUNCH(KK)                                                                            \
  do {                                                                                        \
    PHC_HIP(hipFuncSetAttribute((const void *)qrbs_solve_kernel<KK, CX>,                     \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)(per * wv))); \
    hipLaunchKernelGGL((qrbs_solve_kernel<KK, CX>), dim3(grid), dim3(64 * wv), per * wv, st,  \
                       n, degp1, tailidx, nbatch, mat, rhs, sol, Q, R, flags);                \
  } while (0)
  if (K == 1 && !CX) LAUNCH(1);
  else if (K == 2) LAUNCH(2);
  else LAUNCH(4);
#undef LAUNCH
  PHC_HIP(hipGetLastError());
  return 0;
}

template <bool CX>
int linear_residue_batch(int K, int n, int degp1, int tailidx, int nbatch, const double *mat,
                         const double *rhs, const double *sol, double *res, double *resmax,
                         void *stream, const char *fn) {
  // complex octo-double (K = 8) is refused: its first device run stalled
  // (a launch of houseqr_kernel<8, true> that did not return), cause not
  // established
  PHC_REQUIRE(CX ? (K == 2 || K == 4) : (K == 1 || K == 2 || K == 4),
              std::string(fn) + (CX ? ": K must be 2 or 4" : ": K must be 1, 2 or 4"));
  PHC_REQUIRE(n >= 1 && degp1 >= 1 && nbatch >= 0 && tailidx >= 0,
              std::string(fn) + ": bad sizes");
  PHC_REQUIRE(mat && rhs && sol && res && resmax, std::string(fn) + ": null array");
  if (nbatch == 0) return 0;
  const int wv = 4, grid = (nbatch + wv - 1) / wv;
  hipStream_t st = (hipStream_t)stream;
#define LAUNCH(KK)                                                                            \
  hipLaunchKernelGGL((linear_residue_kernel<KK, CX>), dim3(grid), dim3(64 * wv), 0, st, n,    \
                     degp1, tailidx, nbatch, mat, rhs, sol, res, resmax)
  if (K == 1 && !CX) LAUNCH(1);
  else if (K == 2) LAUNCH(2);
  else LAUNCH(4);
#undef LAUNCH
  PHC_HIP(hipGetLastError());
  return 0;
}

}  // namespace

extern "C" {

int phc_row_newton(phc_rowsys *s, int K, int deg, int nbsteps, int nsys, const double *cst,
                   int cst_shared, const double *cff, int cff_shared, double *x, int *steps,
                   int *wdeg, int *tail, int *up, int *bs, double *history, double *Q, double *R,
                   void *stream) {
  return row_newton<false>(s, K, deg, nbsteps, nsys, cst, cst_shared, cff, cff_shared, nullptr,
                           0, x, steps, wdeg, tail, up, bs, history, Q, R, stream,
                           "phc_row_newton");
}

int phc_column_newton(phc_rowsys *s, int K, int deg, int nbsteps, int nsys, const double *cff,
                      int cff_shared, const double *mb, int mb_shared, double *x, int *steps,
                      int *wdeg, int *tail, int *up, int *bs, double *history, double *Q,
                      double *R, void *stream) {
  PHC_REQUIRE(s && s->S.column, "phc_column_newton: not a column system (phc_colsys_create)");
  PHC_REQUIRE(mb, "phc_column_newton: null right-hand side");
  // a monomial system's coefficients are the unit series
  // (dbl2_unit_series_vector at each step, Newton/dbl2_newton_method.cpp:292)
  return row_newton<false>(s, K, deg, nbsteps, nsys, nullptr, 0, s->nbrcol == 1 ? nullptr : cff,
                           cff_shared, mb, mb_shared, x, steps, wdeg, tail, up, bs, history, Q, R,
                           stream, "phc_column_newton");
}

int phc_cmplx_row_newton(phc_rowsys *s, int K, int deg, int nbsteps, int nsys, const double *cst,
                         int cst_shared, const double *cff, int cff_shared, double *x,
                         int *steps, int *wdeg, int *tail, int *up, int *bs, double *history,
                         double *Q, double *R, void *stream) {
  return row_newton<true>(s, K, deg, nbsteps, nsys, cst, cst_shared, cff, cff_shared, nullptr, 0,
                          x, steps, wdeg, tail, up, bs, history, Q, R, stream,
                          "phc_cmplx_row_newton");
}

int phc_houseqr_batch(int K, int n, int nbatch, const double *A, double *Q, double *R,
                      void *stream) {
  return houseqr_batch<false>(K, n, nbatch, A, Q, R, stream, "phc_houseqr_batch");
}

int phc_cmplx_houseqr_batch(int K, int n, int nbatch, const double *A, double *Q, double *R,
                            void *stream) {
  return houseqr_batch<true>(K, n, nbatch, A, Q, R, stream, "phc_cmplx_houseqr_batch");
}

int phc_qrbs_solve_batch(int K, int n, int degp1, int tailidx, int nbatch, const double *mat,
                         double *rhs, double *sol, double *Q, double *R, int *flags,
                         void *stream) {
  return qrbs_solve_batch<false>(K, n, degp1, tailidx, nbatch, mat, rhs, sol, Q, R, flags,
                                 stream, "phc_qrbs_solve_batch");
}

int phc_cmplx_qrbs_solve_batch(int K, int n, int degp1, int tailidx, int nbatch,
                               const double *mat, double *rhs, double *sol, double *Q, double *R,
                               int *flags, void *stream) {
  return qrbs_solve_batch<true>(K, n, degp1, tailidx, nbatch, mat, rhs, sol, Q, R, flags, stream,
                                "phc_cmplx_qrbs_solve_batch");
}

int phc_linear_residue_batch(int K, int n, int degp1, int tailidx, int nbatch,
                             const double *mat, const double *rhs, const double *sol,
                             double *res, double *resmax, void *stream) {
  return linear_residue_batch<false>(K, n, degp1, tailidx, nbatch, mat, rhs, sol, res, resmax,
                                     stream, "phc_linear_residue_batch");
}

int phc_cmplx_linear_residue_batch(int K, int n, int degp1, int tailidx, int nbatch,
                                   const double *mat, const double *rhs, const double *sol,
                                   double *res, double *resmax, void *stream) {
  return linear_residue_batch<true>(K, n, degp1, tailidx, nbatch, mat, rhs, sol, res, resmax,
                                    stream, "phc_cmplx_linear_residue_batch");
}

}  // extern "C"
