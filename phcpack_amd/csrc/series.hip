// Batched multiple-double arithmetic, truncated power series products and
// polynomial evaluation/differentiation at power series on gfx950.
//
// Reference counterparts:
//   elementwise dd/qd/od ops   Norms/*_gpufun.cu (ddg_*, qdg_*, odg_*)
//   series product             GPU_dbl2_product, Convolutions/dbl2_convolutions_kernels.cu:372
//   polynomial eval/diff       GPU_dbl2_poly_evaldiff, Polynomials/dbl2_polynomials_kernels.cu:1577
// The reference launches one block of deg+1 threads per product and one
// polynomial per call; here one launch covers a batch of independent
// products, and a polynomial takes two, one over all its monomials at a batch
// of instances (one per power-series Newton system or path), one over its
// sums; the plan holding the monomial structure and coefficients stays
// resident on the device.  The order of the
// multiple-double operations per coefficient is that of the reference host
// code (CPU_dbl2_product, CPU_dbl2_poly_speel), so results are bit-identical
// to it.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstring>
#include <vector>
#include "common.hpp"
#include "mdtypes.hpp"
#include "../../include/phcmd.h"

using namespace md;

namespace {

// c ? a : b, limb by limb
__device__ __forceinline__ double pick_real(bool c, double a, double b) { return c ? a : b; }
template <int K> __device__ __forceinline__ mdr<K> pick_real(bool c, const mdr<K> &a, const mdr<K> &b) {
  mdr<K> r;
#pragma unroll
  for (int i = 0; i < K; ++i) r.x[i] = c ? a.x[i] : b.x[i];
  return r;
}

// number traits: real (K limbs) or complex (2K planes)
template <int K, bool CPLX> struct Num;
template <int K> struct Num<K, false> {
  typedef typename RealT<K>::type V;
  static constexpr int P = K;
  static constexpr bool CX = false;
  __device__ static V load(const double *p, size_t s, size_t j) { return R<K>::load(p, s, j); }
  __device__ static void store(double *p, size_t s, size_t j, const V &v) { R<K>::store(p, s, j, v); }
  __device__ static V mul(const V &a, const V &b) { return md::mul(a, b); }
  __device__ static void mac(V &c, const V &a, const V &b) { c = md::add(c, md::mul(a, b)); }
  __device__ static void inc(V &c, const V &a) { c = md::add(c, a); }
  __device__ static V zero() { return R<K>::zero(); }
  __device__ static V pick(bool c, const V &a, const V &b) { return pick_real(c, a, b); }
  __device__ static V pick_v(bool c, const V &a, const V &b) { return pick_real(c, a, b); }
};
template <int K> struct Num<K, true> {
  typedef cplx<K> V;
  static constexpr int P = 2 * K;
  static constexpr bool CX = true;
  __device__ static V load(const double *p, size_t s, size_t j) { return C<K>::load(p, s, j); }
  __device__ static void store(double *p, size_t s, size_t j, const V &v) { C<K>::store(p, s, j, v); }
  __device__ static V mul(const V &a, const V &b) { return C<K>::mul(a, b); }
  __device__ static void mac(V &c, const V &a, const V &b) { C<K>::mac(c, a, b); }
  __device__ static void inc(V &c, const V &a) { c = C<K>::add(c, a); }
  __device__ static V zero() { return C<K>::zero(); }
  template <class T> __device__ static T pick(bool c, const T &a, const T &b) { return pick_real(c, a, b); }
  __device__ static V pick_v(bool c, const V &a, const V &b) {
    V v;
    v.re = pick_real(c, a.re, b.re);
    v.im = pick_real(c, a.im, b.im);
    return v;
  }
};

// ----------------------------------------------------------- elementwise --

template <int K>
__global__ void __launch_bounds__(256) md_batch_kernel(int op, int n, const double *a, const double *b, double *c) {
  typedef typename RealT<K>::type T;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
    T x = R<K>::load(a, n, j), z;
    T y = (op < 4) ? R<K>::load(b, n, j) : R<K>::zero();
    if (op == 0) z = md::add(x, y);
    else if (op == 1) z = md::sub(x, y);
    else if (op == 2) z = md::mul(x, y);
    else if (op == 3) z = md::div(x, y);
    else z = R<K>::sqrt(x);
    R<K>::store(c, n, j, z);
  }
}

// -------------------------------------------------------- series product --

// coefficient k of x*y: x_0*y_k, then += x_i*y_{k-i} for i = 1..k
template <class N>
__device__ typename N::V coef_product(const double *x, size_t sx, size_t xo, const double *y,
                                      size_t sy, size_t yo, int k) {
  typename N::V acc = N::mul(N::load(x, sx, xo), N::load(y, sy, yo + k));
  for (int i = 1; i <= k; ++i) N::mac(acc, N::load(x, sx, xo + i), N::load(y, sy, yo + k - i));
  return acc;
}

// acc = x*y when first, else acc + x*y, each in the order of N::mul and N::mac
template <class N>
__device__ __forceinline__ void mac_or_mul(typename N::V &acc, bool first, const typename N::V &x,
                                           const typename N::V &y) {
  if constexpr (N::CX) {
    const auto re1 = md::mul(x.re, y.re), im1 = md::mul(x.im, y.re);
    const auto re = N::pick(first, re1, md::add(acc.re, re1));
    const auto im = N::pick(first, im1, md::add(acc.im, im1));
    acc.re = md::sub(re, md::mul(x.im, y.im));
    acc.im = md::add(im, md::mul(x.re, y.im));
  } else {
    const auto p = md::mul(x, y);
    acc = N::pick(first, p, md::add(acc, p));
  }
}

// Two truncated products at once by the D lanes of a group: lane k forms
// coefficient k of x1*y1, then coefficient D-1-k of x2*y2 (no second product:
// any rows, the result unused), D + 1 multiply-adds on every lane, where one
// lane per coefficient of one product leaves half of the lanes idle on
// average.  The terms of a coefficient keep the order of coef_product.  In
// double-double a sum starts from zero, to which the first product (never -0 in
// its head) is added without a change.  x1, ...: offsets of the rows in p, numbers with their
// limbs side by side.
template <class N>
__device__ __forceinline__ void product_pair(const double *p, int x1, int y1, int x2, int y2, int D, int k,
                                             typename N::V &r1, typename N::V &r2) {
  constexpr int P = N::P, U = P <= 4 ? 2 : 1;
  constexpr bool from_zero = (N::CX ? P / 2 : P) == 2;
  const double *px = p + x1 * P, *py = p + (y1 + k) * P, *const px2 = p + x2 * P,
               *const py2 = p + (y2 + D - 1 - k) * P;
  typename N::V acc = N::zero(), turned = N::zero();
  bool first = true;
#pragma unroll U
  for (int it = 0; it <= D; ++it) {
    const typename N::V x = N::load(px, 1, 0), y = N::load(py, 1, 0);
    if constexpr (from_zero) N::mac(acc, x, y);
    else mac_or_mul<N>(acc, first, x, y);
    const bool turn = it == k;
    turned = N::pick_v(turn, acc, turned);
    if constexpr (from_zero) acc = N::pick_v(turn, N::zero(), acc);
    first = turn;
    px = turn ? px2 : px + P;
    py = turn ? py2 : py - P;
  }
  r1 = turned;
  r2 = acc;
}

// z[b] = x[b]*y[b] for b < nbatch; arrays [P][nbatch][D]
template <int K, bool CPLX>
__global__ void __launch_bounds__(256) product_kernel(int D, int nbatch, const double *x, const double *y, double *z) {
  typedef Num<K, CPLX> N;
  const size_t s = (size_t)nbatch * D;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < s;
       t += (size_t)gridDim.x * blockDim.x) {
    const size_t b = t / D;
    const int k = (int)(t % D);
    N::store(z, s, t, coef_product<N>(x, s, b * D, y, s, b * D, k));
  }
}

// The same for many products: D lanes take two of them, staged through LDS (4
// rows of D numbers), in blocks of gpb groups.  4096 complex quad-double
// products of degree 31: 155 us with a lane per coefficient, whose loads are
// from global memory and whose lanes idle half of the time, 85 us here.
template <int K, bool CPLX>
__global__ void __launch_bounds__(256) product_pair_kernel(int D, int nbatch, const double *__restrict__ x,
                                       const double *__restrict__ y, double *__restrict__ z, int gpb) {
  typedef Num<K, CPLX> N;
  extern __shared__ __align__(16) double lds[];
  const size_t s = (size_t)nbatch * D;
  const int grp = threadIdx.x / D, k = threadIdx.x % D;
  const size_t b = 2 * ((size_t)blockIdx.x * gpb + grp);
  const bool on = grp < gpb && b < (size_t)nbatch, two = on && b + 1 < (size_t)nbatch;
  double *w = lds + (size_t)grp * 4 * D * N::P;
  if (on) {
    N::store(w + k * N::P, 1, 0, N::load(x, s, b * D + k));
    N::store(w + (D + k) * N::P, 1, 0, N::load(y, s, b * D + k));
    N::store(w + (2 * D + k) * N::P, 1, 0, two ? N::load(x, s, b * D + D + k) : N::zero());
    N::store(w + (3 * D + k) * N::P, 1, 0, two ? N::load(y, s, b * D + D + k) : N::zero());
  }
  __syncthreads();
  if (!on) return;
  typename N::V r1, r2;
  product_pair<N>(w, 0, D, 2 * D, 3 * D, D, k, r1, r2);
  N::store(z, s, b * D + k, r1);
  if (two) N::store(z, s, b * D + 2 * D - 1 - k, r2);
}

// ------------------------------------------------ polynomial eval / diff --

// The contributions of every monomial at every instance: monomial i's value
// and its derivatives with respect to idx[idxptr[i]..], in slots idxptr[i]+i
// (the value) and the nvr[i] slots after it, in contrib [P][nslots][nb][D]
// for the nb instances b0, b0+1, ... of input [P][nbatch][dim][D].
//   D lanes (lane k) per monomial and instance; the forward and the backward
// chain of CPU_dbl2_speel advance together, one product_pair a level, then the
// cross products in pairs: nv + (nv-2)/2 levels for nv >= 3.  Operands (the
// variables X, the coefficient C, the chains F and B) are 3 nvmax - 2 rows (at
// least 2) of the group's work area, in LDS or (LW false) in global memory.
//   One block walking through all monomials of an instance, the chains in
// global memory, took 16.4 ms for one double-double polynomial of 560
// monomials at degree 31 (29 us a monomial, two of the chip's wavefronts
// busy); monomials are independent, and only the sums over them have an
// order, which poly_sum_kernel keeps: 74 us for the two kernels.  1021
// instances of 10 complex quad-double monomials of 4 variables at degree 15:
// 3.59 -> 0.88 ms (16 TFLOP/s of FP64 operations; the FP64 pipes, about 40
// TFLOP/s without fused multiply-adds, bound it).
template <int K, bool CPLX, bool LW>
__global__ void __launch_bounds__(256) poly_terms_kernel(int dim, int nbr, int D, int nvmax, int rows,
                                     const int *__restrict__ nvr, const int *__restrict__ idxptr,
                                     const int *__restrict__ idx, const double *__restrict__ cff,
                                     int nbatch, int b0, int nb, const double *__restrict__ input,
                                     double *__restrict__ contrib, size_t sT, double *work, int gpb) {
  typedef Num<K, CPLX> N;
  typedef typename N::V V;
  extern __shared__ __align__(16) double lds[];
  const int grp = threadIdx.x / D, k = threadIdx.x % D;
  const size_t gid = (size_t)blockIdx.x * gpb + grp;
  const bool on = grp < gpb && gid < (size_t)nbr * nb;
  const int i = on ? (int)(gid / nb) : 0, b = on ? (int)(gid % nb) : 0;
  const int nv = on ? nvr[i] : 0;
  const int *ix = idx + idxptr[i];
  const size_t sX = (size_t)nbatch * dim * D, xb = (size_t)(b0 + b) * dim * D, sC = (size_t)nbr * D;
  // the group's work area: numbers with their limbs side by side
  double *w = LW ? lds + (size_t)grp * rows * D * N::P : work + gid * rows * D * N::P;
  auto keep = [&](int row, int q, const V &v) { N::store(w + (row * D + q) * N::P, 1, 0, v); };
  auto slot = [&](int j) { return ((size_t)(idxptr[i] + i + j) * nb + b) * D + k; };
  if (on) {
    for (int j = 0; j < nv; ++j) keep(j, k, N::load(input, sX, xb + (size_t)ix[j] * D + k));
    const V c = N::load(cff, sC, (size_t)i * D + k);
    keep(nv, k, c);
    if (nv == 1) N::store(contrib, sT, slot(1), c);
  }
  const int C = nv, F = nv + 1, B = 2 * nv;  // rows: X 0..nv-1, C, F 0..nv-2, B 0..nv-3
  const int levels = nvmax < 3 ? nvmax : nvmax + (nvmax - 2) / 2;
  for (int t = 0; t < levels; ++t) {
    __syncthreads();
    // the level's products: operand rows, the row to keep a result in and its slot (-1: none)
    int x1 = -1, y1 = 0, x2 = -1, y2 = 0, d1 = -1, d2 = -1, s1 = -1, s2 = -1;
    if (nv == 1 && t == 0) {
      x1 = 0; y1 = C; s1 = 0;
    } else if (nv == 2 && t == 0) {
      x1 = C; y1 = 0; d1 = F; s1 = 2;
      x2 = C; y2 = 1; s2 = 1;
    } else if (nv == 2 && t == 1) {
      x1 = F; y1 = 1; s1 = 0;
    } else if (nv > 2 && t <= nv - 3) {
      x1 = t ? F + t - 1 : C; y1 = t; d1 = F + t;
      x2 = t ? B + t - 1 : nv - 1; y2 = nv - 2 - t; d2 = B + t;
    } else if (nv > 2 && t == nv - 2) {
      x1 = F + t - 1; y1 = t; d1 = F + t; s1 = nv;
      x2 = B + t - 1; y2 = C; s2 = 1;
    } else if (nv > 2 && t == nv - 1) {
      x1 = F + t - 1; y1 = t; s1 = 0;
      x2 = F + t - 2; y2 = t; s2 = nv - 1;
    } else if (nv > 2) {
      const int j = 2 * (t - nv);
      if (j < nv - 3) { x1 = F + j; y1 = B + nv - 4 - j; s1 = j + 2; }
      if (j + 1 < nv - 3) { x2 = F + j + 1; y2 = B + nv - 5 - j; s2 = j + 3; }
    }
    if (x1 >= 0) {
      V r1, r2;
      const bool two = x2 >= 0;
      product_pair<N>(w, x1 * D, y1 * D, two ? x2 * D : 0, y2 * D, D, k, r1, r2);
      if (d1 >= 0) keep(d1, k, r1);
      if (s1 >= 0) N::store(contrib, sT, slot(s1), r1);
      if (two) {
        const int k2 = D - 1 - k;
        if (d2 >= 0) keep(d2, k2, r2);
        if (s2 >= 0) N::store(contrib, sT, slot(s2) + k2 - k, r2);
      }
    }
  }
}

// Output row r < dim: the derivative, the sum of its contributions
// list[lptr[r]..] from zero; row dim: the value, its contributions added to
// the constant; in the order CPU_dbl2_poly_speel adds them (the monomials'
// order), one lane per coefficient.  The chain of additions bounds it: the
// next U contributions are loaded ahead of it.
template <int K, bool CPLX>
__global__ void __launch_bounds__(64) poly_sum_kernel(int dim, int D, const int *__restrict__ lptr,
                                   const int *__restrict__ list, const double *__restrict__ cst,
                                   int nbatch, int b0, int nb, const double *__restrict__ contrib,
                                   size_t sT, double *__restrict__ output) {
  typedef Num<K, CPLX> N;
  typedef typename N::V V;
  constexpr int U = N::P <= 2 ? 8 : N::P <= 4 ? 4 : N::P <= 8 ? 2 : 1;
  const size_t t = (size_t)blockIdx.x * 64 + threadIdx.x, rowlen = (size_t)(dim + 1) * D;
  if (t >= rowlen * nb) return;
  const int k = (int)(t % D), r = (int)(t / D % (dim + 1)), b = (int)(t / rowlen);
  V acc = r == dim ? N::load(cst, D, k) : N::zero();
  const size_t base = (size_t)b * D + k, step = (size_t)nb * D;
  const int e1 = lptr[r + 1];
  int e = lptr[r];
  for (; e + U <= e1; e += U) {
    V v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = N::load(contrib, sT, base + list[e + u] * step);
#pragma unroll
    for (int u = 0; u < U; ++u) N::inc(acc, v[u]);
  }
  for (; e < e1; ++e) N::inc(acc, N::load(contrib, sT, base + list[e] * step));
  N::store(output, (size_t)nbatch * rowlen, (size_t)(b0 + b) * rowlen + (size_t)r * D + k, acc);
}

bool valid_k(int K) { return K == 1 || K == 2 || K == 4 || K == 8; }

}  // namespace

// ================================================================ C-ABI ====

struct phc_poly {
  int K, cplx, dim, nbr, deg;
  int nvmax = 0, nslots = 0;  // most variables of a monomial; contributions of an instance
  int *d_nvr = nullptr, *d_idxptr = nullptr, *d_idx = nullptr;
  int *d_lptr = nullptr, *d_list = nullptr;  // per output row, its contributions in order
  double *d_cst = nullptr, *d_cff = nullptr;
  double *work = nullptr;
  size_t work_cap = 0;
};

extern "C" {

int phc_md_batch(int op, int K, int n, const double *a, const double *b, double *c,
                 void *stream) {
  PHC_REQUIRE(valid_k(K) && K > 1, "phc_md_batch: K must be 2, 4 or 8");
  PHC_REQUIRE(op >= 0 && op <= 4, "phc_md_batch: op must be 0..4");
  PHC_REQUIRE(n >= 0, "phc_md_batch: n < 0");
  if (n == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  const int block = 256, grid = phc::grid_for(n, block);
  if (K == 2) hipLaunchKernelGGL(md_batch_kernel<2>, dim3(grid), dim3(block), 0, st, op, n, a, b, c);
  else if (K == 4) hipLaunchKernelGGL(md_batch_kernel<4>, dim3(grid), dim3(block), 0, st, op, n, a, b, c);
  else hipLaunchKernelGGL(md_batch_kernel<8>, dim3(grid), dim3(block), 0, st, op, n, a, b, c);
  PHC_HIP(hipGetLastError());
  return 0;
}

int phc_series_product(int K, int cplx, int deg, int nbatch, const double *x, const double *y,
                       double *z, void *stream) {
  PHC_REQUIRE(valid_k(K), "phc_series_product: K must be 1, 2, 4 or 8");
  PHC_REQUIRE(deg >= 0 && nbatch >= 0, "phc_series_product: negative size");
  if (nbatch == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  const int D = deg + 1, P = cplx ? 2 * K : K;
  // Pairs of products where the arithmetic outweighs the staging and the four
  // rows of every group fit LDS, else a coefficient per lane.  One lane against
  // pairs, us: real double-double, degree 31, 16 products 7.5 / 5.6, 8192 19.7 /
  // 9.5; quad-double, degree 15, 21.5 / 20.0 and 34.5 / 22.5; but double-double
  // of degree 8, 128 products 3.4 / 3.6, 8192 4.1 / 3.8 (complex 5.1 / 5.5, 7.7 /
  // 6.3) and double of degree 15, 8192 products 3.8 / 4.4.
  const int pblock = D <= 64 ? 64 : (D + 63) / 64 * 64, gpb = pblock / D > 0 ? pblock / D : 1;
  const size_t lds = sizeof(double) * 4 * P * (size_t)D * gpb;
  const bool pairs = D <= 256 && lds <= 64 * 1024 &&
                     (K * D >= 64 || (K > 1 && (size_t)nbatch * D >= 65536));
  const int block = 256, grid = phc::grid_for((size_t)nbatch * D, block);
  const size_t ngrp = ((size_t)nbatch + 1) / 2, pgrid = (ngrp + gpb - 1) / gpb;
  PHC_REQUIRE(!pairs || pgrid < (1u << 31), "phc_series_product: too many products");
#define PL(KK, CC)                                                                               \
  do {                                                                                           \
    if (pairs)                                                                                   \
      hipLaunchKernelGGL((product_pair_kernel<KK, CC>), dim3(pgrid), dim3(pblock), lds, st, D,   \
                         nbatch, x, y, z, gpb);                                                  \
    else                                                                                         \
      hipLaunchKernelGGL((product_kernel<KK, CC>), dim3(grid), dim3(block), 0, st, D, nbatch, x, y, z); \
  } while (0)
  if (!cplx) {
    if (K == 1) PL(1, false); else if (K == 2) PL(2, false); else if (K == 4) PL(4, false); else PL(8, false);
  } else {
    if (K == 1) PL(1, true); else if (K == 2) PL(2, true); else if (K == 4) PL(4, true); else PL(8, true);
  }
#undef PL
  PHC_HIP(hipGetLastError());
  return 0;
}

int phc_poly_create(phc_poly **plan, int K, int cplx, int dim, int nbr, int deg, const int *nvr,
                    const int *idx, const double *cst, const double *cff) {
  PHC_REQUIRE(plan != nullptr, "phc_poly_create: null plan");
  *plan = nullptr;
  PHC_REQUIRE(valid_k(K), "phc_poly_create: K must be 1, 2, 4 or 8");
  PHC_REQUIRE(dim >= 1 && nbr >= 0 && deg >= 0, "phc_poly_create: bad sizes");
  PHC_REQUIRE(deg + 1 <= 256, "phc_poly_create: degree above 255");
  std::vector<int> ptr(nbr + 1, 0);
  for (int i = 0; i < nbr; ++i) {
    PHC_REQUIRE(nvr[i] >= 1 && nvr[i] <= dim, "phc_poly_create: nvr out of range");
    ptr[i + 1] = ptr[i] + nvr[i];
  }
  for (int j = 0; j < ptr[nbr]; ++j)
    PHC_REQUIRE(idx[j] >= 0 && idx[j] < dim, "phc_poly_create: variable index out of range");
  const int P = cplx ? 2 * K : K, D = deg + 1;
  phc_poly *p = new phc_poly();
  p->K = K; p->cplx = cplx; p->dim = dim; p->nbr = nbr; p->deg = deg;
  // the contributions of every output row in the order in which
  // CPU_dbl2_poly_speel adds them: monomial by monomial, two variables as the
  // second, the first; more as the last, the first, the ones between
  std::vector<std::vector<int>> rows(dim + 1);
  for (int i = 0; i < nbr; ++i) {
    const int nv = nvr[i], *ix = idx + ptr[i], s0 = ptr[i] + i;
    if (nv > p->nvmax) p->nvmax = nv;
    rows[dim].push_back(s0);
    if (nv > 1) rows[ix[nv - 1]].push_back(s0 + nv);
    rows[ix[0]].push_back(s0 + 1);
    for (int j = 1; j < nv - 1; ++j) rows[ix[j]].push_back(s0 + 1 + j);
  }
  p->nslots = ptr[nbr] + nbr;
  std::vector<int> lptr(1, 0), list;
  for (const auto &r : rows) {
    list.insert(list.end(), r.begin(), r.end());
    lptr.push_back((int)list.size());
  }
  const size_t ni = (size_t)std::max(ptr[nbr], 1);
  if (hipMalloc(&p->d_nvr, sizeof(int) * std::max(nbr, 1)) != hipSuccess ||
      hipMalloc(&p->d_idxptr, sizeof(int) * (nbr + 1)) != hipSuccess ||
      hipMalloc(&p->d_idx, sizeof(int) * ni) != hipSuccess ||
      hipMalloc(&p->d_lptr, sizeof(int) * lptr.size()) != hipSuccess ||
      hipMalloc(&p->d_list, sizeof(int) * std::max<size_t>(list.size(), 1)) != hipSuccess ||
      hipMalloc(&p->d_cst, sizeof(double) * P * D) != hipSuccess ||
      hipMalloc(&p->d_cff, sizeof(double) * P * std::max(nbr, 1) * D) != hipSuccess) {
    phc_poly_destroy(p);
    phc::set_error("phc_poly_create: device allocation failed");
    return -1;
  }
  if (nbr > 0) {
    PHC_HIP(hipMemcpy(p->d_nvr, nvr, sizeof(int) * nbr, hipMemcpyHostToDevice));
    PHC_HIP(hipMemcpy(p->d_idx, idx, sizeof(int) * ptr[nbr], hipMemcpyHostToDevice));
    PHC_HIP(hipMemcpy(p->d_cff, cff, sizeof(double) * P * nbr * D, hipMemcpyHostToDevice));
    PHC_HIP(hipMemcpy(p->d_list, list.data(), sizeof(int) * list.size(), hipMemcpyHostToDevice));
  }
  PHC_HIP(hipMemcpy(p->d_lptr, lptr.data(), sizeof(int) * lptr.size(), hipMemcpyHostToDevice));
  PHC_HIP(hipMemcpy(p->d_idxptr, ptr.data(), sizeof(int) * (nbr + 1), hipMemcpyHostToDevice));
  PHC_HIP(hipMemcpy(p->d_cst, cst, sizeof(double) * P * D, hipMemcpyHostToDevice));
  *plan = p;
  return 0;
}

int phc_poly_destroy(phc_poly *p) {
  if (!p) return 0;
  hipFree(p->d_nvr); hipFree(p->d_idxptr); hipFree(p->d_idx); hipFree(p->d_lptr); hipFree(p->d_list);
  hipFree(p->d_cst); hipFree(p->d_cff); hipFree(p->work);
  delete p;
  return 0;
}

int phc_poly_evaldiff(phc_poly *p, int nbatch, const double *input, double *output, void *stream) {
  PHC_REQUIRE(p != nullptr, "phc_poly_evaldiff: null plan");
  PHC_REQUIRE(nbatch >= 0, "phc_poly_evaldiff: nbatch < 0");
  if (nbatch == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  const int P = p->cplx ? 2 * p->K : p->K, D = p->deg + 1;
  // operand rows of a monomial; groups of D lanes per block of 64 (or 1)
  const int rows = std::max(3 * p->nvmax - 2, 2);
  const int block = D <= 64 ? 64 : (D + 63) / 64 * 64, gpb = block / D;
  const size_t group = sizeof(double) * P * rows * D;
  // LDS while four or more blocks fit a compute unit; beyond that (many
  // limbs, variables or degrees, where the arithmetic outweighs the loads)
  // the rows are in global memory and registers alone bound the occupancy
  const bool lw = group * gpb <= 40 * 1024;
  // instances per pass: contributions (and rows) up to 256 MiB
  const size_t inst = sizeof(double) * P * p->nslots * D + (lw ? 0 : group * p->nbr);
  size_t nbc = inst ? ((size_t)256 << 20) / inst : (size_t)nbatch;
  nbc = std::min<size_t>(std::max<size_t>(nbc, 1), nbatch);
  const size_t need = inst / sizeof(double) * nbc;
  if (need > p->work_cap) {
    PHC_HIP(hipStreamSynchronize(st));
    hipFree(p->work);
    p->work = nullptr;
    p->work_cap = 0;
    PHC_HIP(hipMalloc(&p->work, sizeof(double) * need));
    p->work_cap = need;
  }
  for (size_t b0 = 0; b0 < (size_t)nbatch; b0 += nbc) {
    const int nb = (int)std::min(nbc, (size_t)nbatch - b0);
    const size_t sT = (size_t)p->nslots * nb * D, ngrp = (size_t)p->nbr * nb;
    const size_t grid1 = (ngrp + gpb - 1) / gpb, grid2 = ((size_t)nb * (p->dim + 1) * D + 63) / 64;
    PHC_REQUIRE(grid1 < (1u << 31) && grid2 < (1u << 31), "phc_poly_evaldiff: too many instances");
#define LP(KK, CC)                                                                               \
  do {                                                                                           \
    if (grid1 && lw)                                                                             \
      hipLaunchKernelGGL((poly_terms_kernel<KK, CC, true>), dim3(grid1), dim3(block),            \
                         group * gpb, st, p->dim, p->nbr, D, p->nvmax, rows, p->d_nvr,           \
                         p->d_idxptr, p->d_idx, p->d_cff, nbatch, (int)b0, nb, input, p->work,   \
                         sT, (double *)nullptr, gpb);                                            \
    else if (grid1)                                                                              \
      hipLaunchKernelGGL((poly_terms_kernel<KK, CC, false>), dim3(grid1), dim3(block), 0, st,    \
                         p->dim, p->nbr, D, p->nvmax, rows, p->d_nvr, p->d_idxptr, p->d_idx,     \
                         p->d_cff, nbatch, (int)b0, nb, input, p->work, sT, p->work + sT * P,    \
                         gpb);                                                                   \
    hipLaunchKernelGGL((poly_sum_kernel<KK, CC>), dim3(grid2), dim3(64), 0, st, p->dim, D,       \
                       p->d_lptr, p->d_list, p->d_cst, nbatch, (int)b0, nb, p->work, sT, output); \
  } while (0)
    if (!p->cplx) {
      if (p->K == 1) LP(1, false); else if (p->K == 2) LP(2, false); else if (p->K == 4) LP(4, false); else LP(8, false);
    } else {
      if (p->K == 1) LP(1, true); else if (p->K == 2) LP(2, true); else if (p->K == 4) LP(4, true); else LP(8, true);
    }
#undef LP
    PHC_HIP(hipGetLastError());
  }
  return 0;
}

}  // extern "C"
