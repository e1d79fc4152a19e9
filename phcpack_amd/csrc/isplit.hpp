// Complex (and real) multiple-double matrix products on the int8 matrix
// cores: every number is cut into signed base-256 digits relative to the
// largest exponent of its row (left operand) or column (right operand), the
// digit products are accumulated without rounding in int32, and the digit
// sums are rounded once to K limbs at the end (the error-free splitting of
// Ozaki, Ogita, Oishi and Rump, "Error-free transformations of matrix
// multiplication by using fast routines of matrix multiplication and its
// applications", Numerical Algorithms 59 (2012)).
//
//   Why: a complex quad-double multiply-add is about 1100 FP64 instructions
// on the vector units, 17 cycles of a SIMD per lane's product.  With S = 32
// digits it is 528 digit pairs times 4 real products, 2112 of the 16384
// multiply-adds of one v_mfma_i32_16x16x64_i8 each: 2 cycles.  The products of
// the 1024 x 1024 complex quad-double factorization in tiles of 128 took 80 ms
// by multiply-adds; by digits 4.8 ms, with 2.2 ms for cutting the operands and
// for the kernels that look for blocks left over.
//
//   Accuracy: a sum is off by at most 2^(1 - 8 S) max|a_i.| max|b_.j| per
// term, plus one rounding to K limbs, where the K-limb multiply-adds are off
// by about 2^-209 (K = 4) or 2^-104 (K = 2) |a_ik| |b_kj| per term.  As long
// as the nonzero numbers of a row or column span at most 2^R, R = 8 S - 1 -
// 209 (K = 4) or - 104 (K = 2) less a few bits, the digits lose nothing
// against the multiply-adds, whatever the numbers meet.  exponent_kernel
// checks that for every 16 rows; output tiles that a row or column beyond it,
// or one with an infinity, a NaN or an extreme exponent, contributes to are
// left to the K-limb kernel, which gets the same flags.
#pragma once
#include <hip/hip_runtime.h>

#include "mdtypes.hpp"

namespace isplit {

using namespace md;

typedef int v4i __attribute__((ext_vector_type(4)));

// S digits of 8 bits in W 64-bit words, IB digits of the left operand held
// in registers at a time (a divisor of S), R the accepted exponent range
template <int K> struct Cut;
template <> struct Cut<2> {
  static constexpr int S = 18, W = 3, IB = 6, R = 36;
};
template <> struct Cut<4> {
  static constexpr int S = 32, W = 4, IB = 8, R = 44;
};

// the digits of a rows x k operand: fragments of 16 rows by 64 k, 1 KiB each
// in the order in which the lanes of a wavefront hold them (lane = 16 (k / 16)
// + row, 16 bytes of consecutive k), [strip][chunk][digit][part]; parts re,
// im, -im (np = 3), re, im (np = 2) or re (np = 1).  e[row]: the exponent, so
// that |x| < 2^(e-1); flag[strip]: not covered.  Rows are padded to 64, k to
// 64.
struct Digits {
  signed char *d;
  int *e, *flag;
  int np, nch;  // parts, chunks of 64 k
};

__host__ __device__ inline int pad64(int n) { return (n + 63) / 64 * 64; }
template <int K> inline size_t digit_bytes(int rows, int k, int np) {
  return (size_t)pad64(rows) * pad64(k) * Cut<K>::S * np;
}

// exponents and flags of 16 rows per block; element (r, k) at p[sr*r + sk*k],
// planes ps apart (RE: K planes, else 2K)
template <int K, bool RE>
__global__ void __launch_bounds__(512)
exponent_kernel(const double *__restrict__ p, size_t ps, long sr, long sk, int rows, int kd,
                int *__restrict__ e, int *__restrict__ flag) {
  __shared__ int hi[512], lo[512];
  __shared__ int bad[16];
  const int t = threadIdx.x;
  // neighbouring lanes read neighbouring addresses
  const int r = sr == 1 ? t & 15 : t >> 5, k0 = sr == 1 ? t >> 4 : t & 31;
  const int row = blockIdx.x * 16 + r;
  int mx = 0, mn = 4096;
  if (row < rows)
    for (int k = k0; k < kd; k += 32) {
      const size_t o = (size_t)(sr * row + sk * k);
      const double re = p[o];
      const int fr = (__double2hiint(re) >> 20) & 0x7ff;
      if (re != 0.0) { mx = max(mx, fr); mn = min(mn, fr); }
      if constexpr (!RE) {
        const double im = p[K * ps + o];
        const int fi = (__double2hiint(im) >> 20) & 0x7ff;
        if (im != 0.0) { mx = max(mx, fi); mn = min(mn, fi); }
      }
    }
  hi[r * 32 + k0] = mx;
  lo[r * 32 + k0] = mn;
  __syncthreads();
  if (t < 16) {
    for (int q = 1; q < 32; ++q) {
      hi[t * 32] = max(hi[t * 32], hi[t * 32 + q]);
      lo[t * 32] = min(lo[t * 32], lo[t * 32 + q]);
    }
    const int h = hi[t * 32], l = lo[t * 32];
    const int rr = blockIdx.x * 16 + t;
    e[rr] = h - 1023 + 2;
    // an exponent far from 1 (products near the ends of the range of a
    // double), infinities and NaN, or a wide row
    bad[t] = h > 0 && (h > 1023 + 400 || l < 1023 - 400 || h - l > Cut<K>::R);
  }
  __syncthreads();
  if (t == 0) {
    int f = 0;
    for (int q = 0; q < 16; ++q) f |= bad[q];
    flag[blockIdx.x] = f;
  }
}

// the digits of |x| < 1/2, x = sum of the limbs times 2^-e, as W words of the
// two's complement of x 2^(8S-1) rounded down per limb, plus 128 in every
// byte: byte b of the words, less 128, is digit S-1-b.  sign -1 negates.
template <int K>
__device__ __forceinline__ void cut(const double *limb, int e, int sign, unsigned long long *v) {
  constexpr int S = Cut<K>::S, W = Cut<K>::W;
#pragma unroll
  for (int w = 0; w < W; ++w) v[w] = 0x8080808080808080ull;
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const long long bits = __double_as_longlong(limb[q]);
    const int f = (int)(bits >> 52) & 0x7ff;
    long long m = bits & 0xfffffffffffffll;
    if (f) m |= 1ll << 52;
    if ((bits < 0) != (sign < 0)) m = -m;
    int sh = (f ? f : 1) - 1075 - e + 8 * S - 1;
    if (sh < 0) {
      m = sh < -62 ? 0 : m >> -sh;
      sh = 0;
    }
    const int base = sh >> 6, r = sh & 63;
    const unsigned long long low = (unsigned long long)m << r;
    const unsigned long long high = (unsigned long long)((m >> (63 - r)) >> 1);
    const unsigned long long ext = (unsigned long long)(m >> 63);
    unsigned long long carry = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const unsigned long long a = w < base ? 0ull : w == base ? low : w == base + 1 ? high : ext;
      const unsigned long long s1 = v[w] + a, s2 = s1 + carry;
      carry = (s1 < a) | (s2 < s1);
      v[w] = s2;
    }
  }
}

// digits of 16 rows x 64 k per block; every lane cuts four consecutive k
template <int K, bool RE>
__global__ void __launch_bounds__(256)
digit_kernel(const double *__restrict__ p, size_t ps, long sr, long sk, int rows, int kd, int conj,
             Digits D) {
  constexpr int S = Cut<K>::S, W = Cut<K>::W;
  const int t = threadIdx.x, strip = blockIdx.y, ch = blockIdx.x;
  const int r = sr == 1 ? t & 15 : t >> 4, q = sr == 1 ? t >> 4 : t & 15;
  const int row = strip * 16 + r, k0 = ch * 64 + 4 * q;
  const int e = D.e[row];
  signed char *out = D.d + ((size_t)strip * D.nch + ch) * S * D.np * 1024 + (q >> 2) * 256 + r * 16 + (q & 3) * 4;
  for (int part = 0; part < D.np; ++part) {
    unsigned long long v[4][W];
    const int sign = part == 0 ? 1 : ((part == 1) == (conj == 0)) ? 1 : -1;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      double limb[K];
      const bool in = row < rows && k0 + a < kd;
      const size_t o = in ? (size_t)(sr * row + sk * (k0 + a)) : 0;
#pragma unroll
      for (int i = 0; i < K; ++i) limb[i] = in ? p[((RE || part == 0) ? i : K + i) * ps + o] : 0.0;
      // limbs that are not those of one K-limb number (a caller's own) may
      // not fit the digits
#pragma unroll
      for (int i = 1; i < K; ++i)
        if (!(fabs(limb[i]) <= fabs(limb[i - 1]) * 0x1p-50)) D.flag[strip] = 1;
      cut<K>(limb, e, sign, v[a]);
    }
    // 4 x 4 byte transposes: digit s of the four numbers into one word
#pragma unroll
    for (int g = 0; g < (S + 3) / 4; ++g) {
      unsigned x[4];
#pragma unroll
      for (int a = 0; a < 4; ++a) x[a] = (unsigned)(v[a][g >> 1] >> (32 * (g & 1)));
      const unsigned lo01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400), hi01 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602);
      const unsigned lo23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400), hi23 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602);
      const unsigned y[4] = {__builtin_amdgcn_perm(lo23, lo01, 0x05040100), __builtin_amdgcn_perm(lo23, lo01, 0x07060302),
                             __builtin_amdgcn_perm(hi23, hi01, 0x05040100), __builtin_amdgcn_perm(hi23, hi01, 0x07060302)};
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int s = S - 1 - (4 * g + b);
        if (s >= 0) *(unsigned *)(out + ((size_t)s * D.np + part) * 1024) = y[b] ^ 0x80808080u;
      }
    }
  }
}

// whether the 64 x 64 block of the result at (i, j) is left to the K-limb kernel
__device__ __forceinline__ bool uncovered(const int *fa, const int *fb, int i, int j) {
  const int a = i / 64 * 4, b = j / 64 * 4;
  return (fa[a] | fa[a + 1] | fa[a + 2] | fa[a + 3] | fb[b] | fb[b + 1] | fb[b + 2] | fb[b + 3]) != 0;
}

// K limbs of sum_d acc[64 d] 2^(-14-8d), |acc| < 2^31: the carries make it
// a two's complement number of 32-bit words (four digits each) below a small
// signed word, whose 48-bit pieces are exact doubles that do not overlap; a
// pass of quick_two_sums up and one down gives the limbs, zeros left out.
template <int K>
__device__ __forceinline__ typename RealT<K>::type digit_sum(const int *acc) {
  constexpr int S = Cut<K>::S, NW = (S + 3) / 4, NT = 1 + (2 * (NW - 1) + 2) / 3;
  unsigned w[NW];
  long long t = 0;
#pragma unroll
  for (int i = NW - 1; i >= 0; --i) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (4 * i + q < S) t += (long long)acc[(4 * i + q) * 64] << (24 - 8 * q);
    w[i] = (unsigned)t;
    t >>= 32;
  }
  double f[NT];
  f[0] = __builtin_fma((double)(int)t, 0x1p32, (double)w[0]) * 0x1p-38;
#pragma unroll
  for (int j = 1; j < NT; ++j) {
    // pieces j = 1, 3, ...: word a and the upper half of the next; j = 2, 4,
    // ...: its lower half and the word after it
    const int a = 1 + 3 * ((j - 1) / 2);
    if (j & 1) {
      const double hi = (double)w[a], lo = a + 1 < NW ? (double)(w[a + 1] >> 16) : 0.0;
      f[j] = __builtin_fma(hi, 0x1p16, lo) * __builtin_ldexp(1.0, -38 - 32 * a - 16);
    } else {
      const double hi = (double)(w[a + 1] & 0xffffu), lo = a + 2 < NW ? (double)w[a + 2] : 0.0;
      f[j] = __builtin_fma(hi, 0x1p32, lo) * __builtin_ldexp(1.0, -38 - 32 * (a + 2));
    }
  }
#pragma unroll
  for (int j = NT - 1; j > 0; --j) f[j - 1] = quick_two_sum(f[j - 1], f[j], f[j]);
  typename RealT<K>::type c = R<K>::zero();
  double s = f[0];
  int p = 0;
#pragma unroll
  for (int j = 1; j < NT; ++j) {
    double e;
    s = quick_two_sum(s, f[j], e);
    const bool next = e != 0.0 && p < K - 1;
    set_limb<K>(c.x, next ? p : K, s);
    p += next;
    s = next ? e : s;
  }
  set_limb<K>(c.x, p, s);
  return c;
}

template <int K> __device__ __forceinline__ typename RealT<K>::type scaled(typename RealT<K>::type a, int e) {
#pragma unroll
  for (int i = 0; i < K; ++i) a.x[i] = ldexp(a.x[i], e);
  return a;
}

// LDS of a block of digit_gemm_kernel
template <int K, bool RE> constexpr size_t gemm_lds() {
  return (size_t)Cut<K>::S * (RE ? 1 : 3) * 1024;
}

// C(i, j) = [C(i, j) +] sum_k A(i, k) B(k, j) from the digits of A's rows and
// B's columns (parts aim, bim, bnim: im of A, im and -im of B, which makes
// conjugates), or with gridDim.z > 1 the partial sums over kchunk k each in
// part[z][i][j], as cgemm_kernel writes them.
//   A wavefront owns 16 x 16 outputs and all S digit sums of their real and
// imaginary parts (2 S accumulators of four registers, one wavefront per SIMD).
// The four wavefronts of a block take four strips of rows with the same
// columns: per 64 k the digits of those columns go to LDS once, and every
// wavefront streams them past IB digits of its rows at a time, the next IB
// loading meanwhile.  At most 1024 k (32 * 1024 * 2 * 2^14 = 2^30) go into an
// int32 before it is rounded out.
template <int K, bool RE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
digit_gemm_kernel(int M, int N, int KD, int kchunk, Digits A, int aim, Digits B, int bim, int bnim,
                  double *Cp, size_t cps, long c0, long c1, int accumulate, double *part, size_t pps) {
  constexpr int S = Cut<K>::S, IB = Cut<K>::IB, NP = RE ? 1 : 3;
  // (wave-uniform, so that the fragments' addresses are scalar)
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int is = blockIdx.y * 4 + wv, js = blockIdx.x;
  if (uncovered(A.flag, B.flag, is * 16, js * 16)) return;
  const int ch0 = blockIdx.z * (kchunk / 64);
  const int ch1 = min(ch0 + kchunk / 64, (KD + 63) / 64);
  // the digits of the columns, 64 k of them; afterwards the digit sums of one
  // of a lane's four outputs on their way to its limbs: the lane's own,
  // indexed at run time, which registers cannot be
  extern __shared__ v4i bs[];
  int (*my)[S][64] = (int (*)[S][64])bs + wv * (RE ? 1 : 2);
  cplx<K> sum[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) sum[r] = C<K>::zero();
  for (int cb = ch0; cb < ch1; cb += 16) {
    v4i accr[S], acci[RE ? 1 : S];
#pragma unroll
    for (int d = 0; d < S; ++d) {
      accr[d] = v4i{0, 0, 0, 0};
      if constexpr (!RE) acci[d] = v4i{0, 0, 0, 0};
    }
    for (int ch = cb; ch < min(cb + 16, ch1); ++ch) {
      const v4i *a = (const v4i *)(A.d + ((size_t)is * A.nch + ch) * S * NP * 1024);
      const v4i *b = (const v4i *)(B.d + ((size_t)js * B.nch + ch) * S * NP * 1024);
      v4i ar[2][IB], ai[2][RE ? 1 : IB];
      __syncthreads();  // every wavefront is done with the LDS
      for (int f = wv; f < S * NP; f += 4)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(b + f * 64 + l),
                                         (__attribute__((address_space(3))) void *)(bs + f * 64), 16, 0, 0);
#pragma unroll
      for (int i = 0; i < IB; ++i) {
        ar[0][i] = (a + i * NP * 64)[l];
        if constexpr (!RE) ai[0][i] = (a + (i * NP + aim) * 64)[l];
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
#pragma unroll
      for (int ib = 0; ib < S; ib += IB) {
        const int h = (ib / IB) & 1;
        v4i br[2], bi[2], bn[2];
        br[0] = bs[l];
        if constexpr (!RE) { bi[0] = bs[bim * 64 + l]; bn[0] = bs[bnim * 64 + l]; }
#pragma unroll
        for (int j = 0; j < S - ib; ++j) {
          // loads stay within a digit of their use: the accumulators take
          // the registers that earlier ones would need
          __builtin_amdgcn_sched_barrier(0);
          const int u = j & 1;
          if (j + 1 < S - ib) {
            br[u ^ 1] = bs[(j + 1) * NP * 64 + l];
            if constexpr (!RE) {
              bi[u ^ 1] = bs[((j + 1) * NP + bim) * 64 + l];
              bn[u ^ 1] = bs[((j + 1) * NP + bnim) * 64 + l];
            }
          }
          if (ib + IB < S && j >= S - ib - 2 * IB && j < S - ib - IB) {
            const int i = j - (S - ib - 2 * IB);  // the rows' next digits, one each time
            ar[h ^ 1][i] = (a + (ib + IB + i) * NP * 64)[l];
            if constexpr (!RE) ai[h ^ 1][i] = (a + ((ib + IB + i) * NP + aim) * 64)[l];
          }
#pragma unroll
          for (int i = 0; i < IB; ++i)
            if (ib + i + j < S)
              accr[ib + i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ar[h][i], br[u], accr[ib + i + j], 0, 0, 0);
          if constexpr (!RE) {
#pragma unroll
            for (int i = 0; i < IB; ++i)
              if (ib + i + j < S)
                acci[ib + i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ar[h][i], bi[u], acci[ib + i + j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < IB; ++i)
              if (ib + i + j < S)
                accr[ib + i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ai[h][i], bn[u], accr[ib + i + j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < IB; ++i)
              if (ib + i + j < S)
                acci[ib + i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ai[h][i], br[u], acci[ib + i + j], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < S; ++d) {
        my[0][d][l] = accr[d][r];
        if constexpr (!RE) my[1][d][l] = acci[d][r];
      }
      __builtin_amdgcn_sched_barrier(0);
      sum[r].re = add(sum[r].re, digit_sum<K>(&my[0][0][l]));
      if constexpr (!RE) sum[r].im = add(sum[r].im, digit_sum<K>(&my[1][0][l]));
    }
  }
  const int j = js * 16 + (l & 15);
  const int eb = B.e[j];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = is * 16 + (l >> 4) * 4 + r;
    if (i >= M || j >= N) continue;
    const int e = A.e[i] + eb;
    cplx<K> v;
    v.re = scaled<K>(sum[r].re, e);
    v.im = RE ? R<K>::zero() : scaled<K>(sum[r].im, e);
    double *out = Cp;
    size_t ops = cps, o = (size_t)(c0 * i + c1 * j);
    if (gridDim.z > 1) {
      out = part;
      ops = pps;
      o = (size_t)blockIdx.z * M * N + (size_t)i * N + j;
    } else if (accumulate) {
      v.re = add(R<K>::load(Cp, cps, o), v.re);
      if constexpr (!RE) v.im = add(R<K>::load(Cp + K * cps, cps, o), v.im);
    }
    R<K>::store(out, ops, o, v.re);
    if constexpr (!RE) R<K>::store(out + K * ops, ops, o, v.im);
  }
}

}  // namespace isplit
