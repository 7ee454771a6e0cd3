// kernels_util.hip -- 6j table, operator arithmetic and norms, normal ordering,
// basis transformation, Hartree-Fock monopoles, synthetic operators, White
// generator, MFMA layout probe.
#include <hip/hip_runtime.h>

#include "internal.hpp"
#include "launch.hpp"

namespace imsrg {

// ---------------------------------------------------------------------------
// double-double arithmetic (Dekker / Knuth two-sum, fma two-product)
struct dd {
  double hi, lo;
};
__device__ __forceinline__ dd dd_quick(double a, double b) {
  double s = a + b;
  return {s, b - (s - a)};
}
__device__ __forceinline__ dd dd_two_sum(double a, double b) {
  double s = a + b;
  double bb = s - a;
  return {s, (a - (s - bb)) + (b - bb)};
}
__device__ __forceinline__ dd dd_add(dd x, dd y) {
  dd s = dd_two_sum(x.hi, y.hi);
  dd t = dd_two_sum(x.lo, y.lo);
  s.lo += t.hi;
  s = dd_quick(s.hi, s.lo);
  s.lo += t.lo;
  return dd_quick(s.hi, s.lo);
}
__device__ __forceinline__ dd dd_neg(dd x) { return {-x.hi, -x.lo}; }
__device__ __forceinline__ dd dd_mul(dd x, dd y) {
  double p = x.hi * y.hi;
  double e = __fma_rn(x.hi, y.hi, -p);
  e += x.hi * y.lo + x.lo * y.hi;
  return dd_quick(p, e);
}
__device__ __forceinline__ dd dd_mul_d(dd x, double y) {
  double p = x.hi * y;
  double e = __fma_rn(x.hi, y, -p);
  e += x.lo * y;
  return dd_quick(p, e);
}
__device__ __forceinline__ dd dd_div(dd x, dd y) {
  double q1 = x.hi / y.hi;
  dd r = dd_add(x, dd_neg(dd_mul_d(y, q1)));
  double q2 = r.hi / y.hi;
  r = dd_add(r, dd_neg(dd_mul_d(y, q2)));
  double q3 = r.hi / y.hi;
  return dd_add(dd_quick(q1, q2), dd{q3, 0.0});
}
__device__ __forceinline__ dd dd_sqrt(dd a) {
  if (a.hi <= 0.0) return {0.0, 0.0};
  double x = sqrt(a.hi);
  dd xx = dd_mul(dd{x, 0.0}, dd{x, 0.0});
  dd r = dd_add(a, dd_neg(xx));
  return dd_two_sum(x, r.hi / (2.0 * x));
}

constexpr int kNFact = 256;

__global__ void k_factorials(dd *f) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    dd v = {1.0, 0.0};
    f[0] = v;
    for (int i = 1; i < kNFact; ++i) {
      v = dd_mul_d(v, (double)i);
      f[i] = v;
    }
  }
}

__device__ __forceinline__ bool tri_ok(int a, int b, int c) {
  return ((a + b + c) & 1) == 0 && c >= abs(a - b) && c <= a + b;
}

// Wigner 6j {a b c; d e f} (doubled arguments), Racah single-sum formula
// (Edmonds eq. 6.3.7) in double-double; replaces gsl_sf_coupling_6j
// (src/AngMom.cc:94-97).
__device__ double sixj_dd(const dd *F, int a, int b, int c, int d, int e, int f) {
  if (!tri_ok(a, b, c) || !tri_ok(a, e, f) || !tri_ok(d, b, f) || !tri_ok(d, e, c)) return 0.0;
  const int tri[4][3] = {{a, b, c}, {a, e, f}, {d, b, f}, {d, e, c}};
  // product of the four triangle coefficients, each formed as its own ratio
  // (at most 1): the four denominators multiplied first overflow a double
  // for j = 29/2, J = 29 (emax = 14)
  dd d2 = {1.0, 0.0};
  for (int k = 0; k < 4; ++k) {
    int x = tri[k][0], y = tri[k][1], z = tri[k][2];
    const dd num = dd_mul(dd_mul(F[(x + y - z) / 2], F[(x - y + z) / 2]), F[(-x + y + z) / 2]);
    d2 = dd_mul(d2, dd_div(num, F[(x + y + z) / 2 + 1]));
  }
  dd pref = dd_sqrt(d2);
  const int al[4] = {(a + b + c) / 2, (a + e + f) / 2, (d + b + f) / 2, (d + e + c) / 2};
  const int be[3] = {(a + b + d + e) / 2, (b + c + e + f) / 2, (a + c + d + f) / 2};
  int tmin = max(max(al[0], al[1]), max(al[2], al[3]));
  int tmax = min(min(be[0], be[1]), be[2]);
  dd sum = {0.0, 0.0};
  for (int t = tmin; t <= tmax; ++t) {
    dd dn = F[t - al[0]];
    for (int k = 1; k < 4; ++k) dn = dd_mul(dn, F[t - al[k]]);
    for (int k = 0; k < 3; ++k) dn = dd_mul(dn, F[be[k] - t]);
    dd term = dd_div(F[t + 1], dn);
    if (t & 1) term = dd_neg(term);
    sum = dd_add(sum, term);
  }
  dd r = dd_mul(pref, sum);
  return r.hi + r.lo;
}

__global__ __launch_bounds__(256) void k_sixj_table(const dd *F, double *table, double *tableQ, int d1, int d2,
                                                   long total) {
  for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
    long r = idx;
    const int J6 = r % d2; r /= d2;
    const int i5 = r % d1; r /= d1;
    const int i4 = r % d1; r /= d1;
    const int J3 = r % d2; r /= d2;
    const int i2 = r % d1; r /= d1;
    const int i1 = (int)r;
    const double v = sixj_dd(F, 2 * i1 + 1, 2 * i2 + 1, 2 * J3, 2 * i4 + 1, 2 * i5 + 1, 2 * J6);
    table[idx] = v;
    // the inverse Pandya copy holds the weights (2 J6 + 1) {...}, and 0 where
    // |6j| < 1e-8, the values whose terms the reference skips (src/Commutator.cc:1564-1572,
    // 1593-1604)
    tableQ[sixjQ_index(d1, d2, 2 * i1 + 1, 2 * i2 + 1, J3, 2 * i4 + 1, 2 * i5 + 1, J6)] =
        fabs(v) >= 1e-8 ? (2 * J6 + 1) * v : 0.0;
  }
}

hipError_t launch_sixj_table(double *table, double *tableQ, int d1, int d2, hipStream_t s) {
  if (4 * (d1 - 1) + 4 > kNFact - 4) return hipErrorInvalidValue;
  dd *F = nullptr;
  hipError_t e = hipMalloc(&F, sizeof(dd) * kNFact);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_factorials, dim3(1), dim3(64), 0, s, F);
  long total = (long)d1 * d1 * d2 * d1 * d1 * d2;
  int blocks = (int)std::min<long>((total + 255) / 256, 65536);
  hipLaunchKernelGGL(k_sixj_table, dim3(blocks), dim3(256), 0, s, F, table, tableQ, d1, d2, total);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  e = hipStreamSynchronize(s);
  (void)hipFree(F);
  return e;
}

// ---------------------------------------------------------------------------
// y = z + a x; z may be y
__global__ __launch_bounds__(256) void k_axpy(double *y, const double *z, double a, const double *x, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    double t = a * x[i];  // (a*x) formed first, then added (Operator operator* then +=)
    y[i] = z[i] + t;
  }
}
__global__ __launch_bounds__(256) void k_scale(double *y, double a, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) y[i] *= a;
}
// y[i] = v (clears memory that may hold NaN or Inf, which a scale by 0 keeps)
__global__ __launch_bounds__(256) void k_fill(double *y, double v, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) y[i] = v;
}
static int grid_for(long n) { return (int)std::max<long>(1, std::min<long>((n + 255) / 256, 8192)); }
hipError_t launch_fill(double *y, double v, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(256), 0, s, y, v, n);
  return hipGetLastError();
}
hipError_t launch_axpy(double *y, const double *z, double a, const double *x, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy, dim3(grid_for(n)), dim3(256), 0, s, y, z, a, x, n);
  return hipGetLastError();
}
hipError_t launch_scale(double *y, double a, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_scale, dim3(grid_for(n)), dim3(256), 0, s, y, a, n);
  return hipGetLastError();
}

// One pass over an operator buffer x with the partial sums of its norm: OP 0 the sums
// alone, OP 1 y = z + a x beside them (z is y, or Op at the first term: the BCH_Transform
// step, src/BCH.cc:176-191), OP 2 y = x (a copy).  Block b < nblk2 takes the b-th contiguous chunk of the two-body arena,
// each word with its channel's weight (2J+1)^2; blocks nblk2 .. nblk2 + nblk1 - 1 share the
// one-body part (weights 2 j_p + 1), the first of them the words around the two parts.
// Bound by HBM at large sizes: a block has four 16-byte loads per thread in flight (one
// 8-byte load each: the norm 101 us for 293 MB at emax = 10, and a separate device copy about
// as long again).  At small sizes by the longest chain of loads in a block: with one block
// for the one-body part and the channels of a chunk one after the other, axpy and norm took
// 37 us at emax = 7 (22 MB) and 27 us at emax = 6, now 16 and 9 us.
constexpr int kNormCh = 640;  // channels whose offsets fit in the kernel's LDS list
template <int OP>
__global__ __launch_bounds__(256) void k_norm_pass(const BasisDev *bd, double *y, const double *z, double a,
                                                   const double *x, double *part, int nblk2, int nblk1) {
  const BasisDev &B = *bd;
  __shared__ double red[4];
  __shared__ long s_off[kNormCh];
  double acc = 0.0;
  constexpr int U = 4;
  if ((int)blockIdx.x >= nblk2) {
    auto put = [&](long e, double v) {  // one word of y
      if (OP == 1) {
        double t = a * v;  // (a x) formed first, then added (Operator operator* then +=)
        y[e] = z[e] + t;
      }
      if (OP == 2) y[e] = v;
    };
    const int b1 = blockIdx.x - nblk2;
    const long n1 = (long)B.norb * B.norb;
    // the zero-body and padding words around the one-body block and after the two-body arena
    const long rg[3][2] = {{0, B.one_off}, {B.one_off + n1, B.two_off}, {B.two_off + B.tbsize, B.opsize}};
    if (OP != 0 && b1 == 0)
      for (int g = 0; g < 3; ++g)
        for (long e = rg[g][0] + threadIdx.x; e < rg[g][1]; e += blockDim.x) put(e, x[e]);
    const double *x1 = x + B.one_off;
    double *y1 = OP ? y + B.one_off : nullptr;
    const double *z1 = OP == 1 ? z + B.one_off : nullptr;
    for (long q = (long)b1 * blockDim.x + threadIdx.x; q < n1; q += (long)U * nblk1 * blockDim.x) {
      double v[U], w[U], o[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long e = min(q + (long)u * nblk1 * blockDim.x, n1 - 1);
        v[u] = x1[e];
        w[u] = B.w1norm[e];
        if (OP == 1) o[u] = z1[e];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long e = q + (long)u * nblk1 * blockDim.x;
        if (e >= n1) break;
        acc += v[u] * v[u] * w[u];
        if (OP == 1) {
          double t = a * v[u];
          y1[e] = o[u] + t;
        }
        if (OP == 2) y1[e] = v[u];
      }
    }
  } else {
    const double *two = x + B.two_off;
    double *y2 = OP ? y + B.two_off : nullptr;
    const double *z2 = OP == 1 ? z + B.two_off : nullptr;
    const long tb = B.tbsize, chunk = (tb + nblk2 - 1) / nblk2;
    const long c0 = (long)blockIdx.x * chunk, c1 = min(c0 + chunk, tb);
    // the channels that the chunk overlaps: lo .. hi
    const int nch = B.nch;
    int lo = -1, hi = -1;
    for (int c = 0; c < nch; c += blockDim.x) {
      const int ch = c + threadIdx.x;
      const long off = ch < nch ? B.ch_off[ch] : tb;
      if (ch < min(nch, kNormCh)) s_off[ch] = off;
      lo += __syncthreads_count(ch < nch && off <= c0);
      hi += __syncthreads_count(ch < nch && off < c1);
    }
    auto weight = [](int ch) { return (double)((2 * (ch / 6) + 1) * (2 * (ch / 6) + 1)); };
    auto offset = [&](int ch) -> long { return ch < kNormCh ? s_off[ch] : B.ch_off[ch]; };
    const double wlo = weight(max(lo, 0));
    // pairs of words at even offsets (the arena is 64-byte aligned), clamped into [c0, c1):
    // a pair across an end counts its inner word only
    for (long q = (c0 & ~1L) + 2 * (long)threadIdx.x; q < c1; q += 2 * U * (long)blockDim.x) {
      double2 v[U], o[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long e = min(q + 2 * u * (long)blockDim.x, (c1 - 1) & ~1L);
        v[u] = *reinterpret_cast<const double2 *>(two + e);
        if (OP == 1) o[u] = *reinterpret_cast<const double2 *>(z2 + e);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long e = q + 2 * u * (long)blockDim.x;
        const bool m0 = e < c1 && e >= c0, m1 = e + 1 < c1;
        double w0 = wlo, w1 = wlo;
        if (lo < hi) {  // the words' channels
          int a0 = lo, a1 = hi;
          while (a0 < a1) {
            const int mid = (a0 + a1 + 1) >> 1;
            if (offset(mid) <= max(e, c0)) a0 = mid; else a1 = mid - 1;
          }
          w0 = weight(a0);
          while (a0 < hi && offset(a0 + 1) <= e + 1) ++a0;
          w1 = weight(a0);
        }
        if (m0) acc += w0 * (v[u].x * v[u].x);
        if (m1) acc += w1 * (v[u].y * v[u].y);
        if (OP == 0) continue;
        double2 r = v[u];
        if (OP == 1) {
          double t0 = a * v[u].x, t1 = a * v[u].y;
          r.x = o[u].x + t0;
          r.y = o[u].y + t1;
        }
        if (m0 && m1)
          *reinterpret_cast<double2 *>(y2 + e) = r;
        else if (m0)
          y2[e] = r.x;
        else if (m1)
          y2[e + 1] = r.y;
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// The norm's two sums into out[0..1]; with seq != 0, out is host memory, and seq goes
// into *done after them, so that the host can read the sums without a copy and without
// waiting for the stream.
__global__ __launch_bounds__(256) void k_norm_final(const double *part, int nblk2, int nblk1, double *out,
                                                    unsigned long long *done, unsigned long long seq) {
  __shared__ double red[4];
  double acc = 0.0, one = (int)threadIdx.x < nblk1 ? part[nblk2 + threadIdx.x] : 0.0;
  for (int i = threadIdx.x; i < nblk2; i += blockDim.x) acc += part[i];
  for (int o = 32; o > 0; o >>= 1) {
    acc += __shfl_down(acc, o, 64);
    one += __shfl_down(one, o, 64);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    out[0] = one;  // nblk1 <= 64: the first wave's
    out[1] = (red[0] + red[1]) + (red[2] + red[3]);
    if (seq) {
      __threadfence_system();
      __hip_atomic_store(done, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// Operator::DoNormalOrdering2 of a scalar operator (src/Operator.cc:461-579) in
// place, sign +1 (normal ordering) or -1 (undoing it), over the reference's holes.
// Zero-body part (:467-490): E0 += sign sum_k (2j_k+1) n_k h_kk + sum_{k<=l} sum_J
// (2J+1) n_k n_l V^J_{kl,kl} (normalized), one thread per hole pair and a
// fixed-order block sum; it reads the one-body diagonal before k_no_one changes it.
__global__ __launch_bounds__(256) void k_no_zero(const BasisDev *Bp, double *op, int sign) {
  __shared__ double red[4];
  const BasisDev &B = *Bp;
  const int norb = B.norb, nh = B.nholes;
  const double *one = op + B.one_off, *two = op + B.two_off;
  double acc = 0.0;
  for (int t = threadIdx.x; t < nh * nh; t += blockDim.x) {
    const int ik = t / nh, il = t - ik * nh;
    const int k = B.holes[ik], l = B.holes[il];
    if (ik == il) acc += (B.j2[k] + 1) * sign * B.occ[k] * one[(long)k * norb + k];
    if (l < k) continue;
    const int par = (B.l[k] + B.l[l]) & 1, tz = (B.tz2[k] + B.tz2[l]) / 2;
    const int kl = ket_index(norb, k, l);
    for (int J = abs(B.j2[k] - B.j2[l]) / 2; J <= (B.j2[k] + B.j2[l]) / 2; ++J) {
      const int i = B.kmapT[(long)J * B.nkets + kl];  // -1: (k,k) at odd J
      if (i < 0) continue;
      const int ch = 6 * J + 2 * (tz + 1) + par, n = B.ch_n[ch];
      acc += (2 * J + 1) * B.occ[k] * B.occ[l] * two[B.ch_off[ch] + (long)i * n + i];
    }
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) op[0] += (red[0] + red[1]) + (red[2] + red[3]);
}

// One-body part (:493-560) and the (anti-)Hermitian completion (Symmetrize /
// AntiSymmetrize, :1797-1830): one wave per pair a <= b of a one-body block, one
// lane per hole h,
//   f_ab += sign sum_J (2J+1)/(2j_a+1) n_h V~^J_{ah,bh}
// with the tilde element (sqrt 2 per ket with equal orbits, (-1)^{(j_p+j_q)/2+1+J}
// per swapped ket), summed over the lanes in a fixed order.  The sum is skipped
// when the two-body norm (n2sq = its square, on the device) is at most 1e-7.
__global__ __launch_bounds__(256) void k_no_one(const BasisDev *Bp, double *op, int sign, int herm,
                                                const double *n2sq) {
  const BasisDev &B = *Bp;
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (p >= B.n1pairs) return;  // wave-uniform
  const int2 pr = B.pairs1[p];
  const int a = pr.x, b = pr.y, norb = B.norb;
  double *one = op + B.one_off;
  const double *two = op + B.two_off;
  double acc = 0.0;
  if (*n2sq > 1e-14) {
    const double w0 = 1.0 / (B.j2[a] + 1.0);  // 1 / (2 j_a + 1)
    for (int ih = lane; ih < B.nholes; ih += 64) {
      const int h = B.holes[ih];
      const int par = (B.l[a] + B.l[h]) & 1, tz = (B.tz2[a] + B.tz2[h]) / 2;
      const int kah = ket_index(norb, min(a, h), max(a, h)), kbh = ket_index(norb, min(b, h), max(b, h));
      const double nrm = (a == h ? 1.4142135623730951 : 1.0) * (b == h ? 1.4142135623730951 : 1.0);
      for (int J = abs(B.j2[a] - B.j2[h]) / 2; J <= (B.j2[a] + B.j2[h]) / 2; ++J) {
        const int i = B.kmapT[(long)J * B.nkets + kah], k = B.kmapT[(long)J * B.nkets + kbh];
        if (i < 0 || k < 0) continue;
        const int ch = 6 * J + 2 * (tz + 1) + par, n = B.ch_n[ch];
        double ph = 1.0;
        if (a > h) ph *= ((B.j2[a] + B.j2[h]) / 2 + 1 + J) & 1 ? -1.0 : 1.0;
        if (b > h) ph *= ((B.j2[b] + B.j2[h]) / 2 + 1 + J) & 1 ? -1.0 : 1.0;
        acc += (2 * J + 1) * w0 * sign * B.occ[h] * (nrm * ph * two[B.ch_off[ch] + (long)k * n + i]);
      }
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  }
  if (lane != 0) return;
  double f = one[(long)b * norb + a] + acc;
  if (herm == -1 && a == b) f = 0.0;
  one[(long)b * norb + a] = f;
  if (a != b) one[(long)a * norb + b] = herm * f;
}

hipError_t launch_normal_order(const BasisDev *bd, const BasisDev &bh, double *op, int sign, int herm,
                               const double *n2sq, hipStream_t s) {
  hipLaunchKernelGGL(k_no_zero, dim3(1), dim3(256), 0, s, bd, op, sign);
  if (bh.n1pairs > 0)
    hipLaunchKernelGGL(k_no_one, dim3((bh.n1pairs + 3) / 4), dim3(256), 0, s, bd, op, sign, herm, n2sq);
  return hipGetLastError();
}

hipError_t launch_norm(const BasisDev *bd, const BasisDev &bh, NormOp op, double *y, const double *z, double a,
                       const double *x, double *partials, int maxpart, double *out, unsigned long long *done,
                       unsigned long long seq, hipStream_t s) {
  // two-body chunks of at least 2048 words, so that small bases do not pay for idle blocks
  const int nblk1 = (int)std::max(1, std::min(32, bh.norb * bh.norb / 1024));
  const int nblk2 = (int)std::max<long>(1, std::min<long>(maxpart - nblk1, (bh.tbsize + 2047) / 2048));
  const dim3 grid(nblk2 + nblk1), blk(256);
  if (op == NormOp::kSum)
    hipLaunchKernelGGL((k_norm_pass<0>), grid, blk, 0, s, bd, y, z, a, x, partials, nblk2, nblk1);
  else if (op == NormOp::kAxpy)
    hipLaunchKernelGGL((k_norm_pass<1>), grid, blk, 0, s, bd, y, z, a, x, partials, nblk2, nblk1);
  else
    hipLaunchKernelGGL((k_norm_pass<2>), grid, blk, 0, s, bd, y, z, a, x, partials, nblk2, nblk1);
  hipLaunchKernelGGL(k_norm_final, dim3(1), dim3(256), 0, s, partials, nblk2, nblk1, out, done, seq);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The two-body basis-change matrix of HartreeFock::TransformToHFBasis
// (src/HartreeFock.cc:942-960), for every channel at once, in the two-body layout:
// element (i, a) of channel ch's block is
//   D(i, a) = C(p, p') C(q, q') + [p != q] Phase_pq(J) C(q, p') C(p, q'),
// times sqrt2 if p == q, divided by sqrt2 if p' == q', for the channel's kets
// i = (p, q) (old basis, rows) and a = (p', q') (new basis, columns);
// Phase_pq(J) = (-1)^{(j_p + j_q)/2 + 1 + J} (src/ModelSpace.hh:72-78).
// C is norb x norb column-major, C(p, p') = <p|p'>.  One thread per element.
__global__ __launch_bounds__(256) void k_hf_D(const BasisDev *bd, const double *C, double *D) {
  const BasisDev &B = *bd;
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= B.tbsize) return;
  int lo = 0, hi = B.nch - 1;  // the last channel starting at or before e holds it
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (B.ch_off[mid] <= e) lo = mid; else hi = mid - 1;
  }
  const int ch = lo, n = B.ch_n[ch], J = ch / 6;
  const long r = e - B.ch_off[ch];
  const int i = (int)(r % n), a = (int)(r / n);
  const int ki = B.ch_kets[B.ch_kstart[ch] + i], ka = B.ch_kets[B.ch_kstart[ch] + a];
  const int p = B.kp[ki], q = B.kq[ki], pp = B.kp[ka], qq = B.kq[ka];
  const long N = B.norb;
  double d = C[p + pp * N] * C[q + qq * N];
  if (p != q) {
    const double ph = (((B.j2[p] + B.j2[q]) / 2 + 1 + J) & 1) ? -1.0 : 1.0;
    double x = C[q + pp * N] * C[p + qq * N];
    d += ph * x;
  }
  if (p == q) d *= 1.4142135623730951;
  if (pp == qq) d /= 1.4142135623730951;
  D[e] = d;
}

// The two-body monopoles of the Hartree-Fock field (HartreeFock::BuildMonopoleV and
// the lookups of UpdateF, src/HartreeFock.cc:250-285, 771-800):
//   W(i a, j b) = sum_J (2J+1) V~^J_{ia,jb}
// with the tilde element (sqrt2 per ket with equal orbits, (-1)^{(j_p+j_q)/2+1+J}
// per swapped ket), J over the couplings of (i, a), summed in ascending J; equal to
// the reference's Vmon / Vmon_exch entry, GetTBMEmonopole times (2j_i+1)(2j_a+1)
// (src/TwoBodyME.cc:614-679).  quads[q] = (i, a, j, b); one thread per quad.
__global__ __launch_bounds__(256) void k_hf_mono(const BasisDev *Bp, const double *op, const int4 *quads, int nq,
                                                 double *W) {
  const BasisDev &B = *Bp;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  const int4 t = quads[q];
  const int i = t.x, a = t.y, j = t.z, b = t.w, norb = B.norb;
  const double *two = op + B.two_off;
  const int par = (B.l[i] + B.l[a]) & 1, tz = (B.tz2[i] + B.tz2[a]) / 2;
  double acc = 0.0;
  if (par == ((B.l[j] + B.l[b]) & 1) && tz == (B.tz2[j] + B.tz2[b]) / 2) {
    const int kia = ket_index(norb, min(i, a), max(i, a)), kjb = ket_index(norb, min(j, b), max(j, b));
    const double nrm = (i == a ? 1.4142135623730951 : 1.0) * (j == b ? 1.4142135623730951 : 1.0);
    for (int J = abs(B.j2[i] - B.j2[a]) / 2; J <= (B.j2[i] + B.j2[a]) / 2; ++J) {
      const int r = B.kmapT[(long)J * B.nkets + kia], c = B.kmapT[(long)J * B.nkets + kjb];
      if (r < 0 || c < 0) continue;
      const int ch = 6 * J + 2 * (tz + 1) + par, n = B.ch_n[ch];
      double ph = 1.0;
      if (i > a) ph *= ((B.j2[i] + B.j2[a]) / 2 + 1 + J) & 1 ? -1.0 : 1.0;
      if (j > b) ph *= ((B.j2[j] + B.j2[b]) / 2 + 1 + J) & 1 ? -1.0 : 1.0;
      acc += (2 * J + 1) * (nrm * ph * two[B.ch_off[ch] + (long)c * n + r]);
    }
  }
  W[q] = acc;
}

hipError_t launch_hf_mono(const BasisDev *bd, const double *op, const int4 *quads, int nq, double *W,
                          hipStream_t s) {
  if (nq > 0) hipLaunchKernelGGL(k_hf_mono, dim3((nq + 255) / 256), dim3(256), 0, s, bd, op, quads, nq, W);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Basis transformation with a basis change C that is block diagonal in (l, j, tz),
// as every Hartree-Fock C is.  D(i, a) is then nonzero only when the kets i and a of
// a channel take their orbits from the same pair of one-body blocks, so after
// grouping each channel's kets by that pair, D is block diagonal with groups of at
// most (block size)^2 kets, and V' = D^T V D is two passes over the channel:
//   T  = V D                              column a of T mixes the columns of V in a's group
//   V' = D^T T = (T^T D)^T                row a of V' mixes the rows of T in a's group
// and the second is the first on T^T, which k_xf_pass<false> stores: U(a, r) = T(r, a), with
// its rows a in the order of the groups (X.g_kets), so that both passes read and the first
// writes runs of consecutive elements.  The second stores V'(a, b) at column b of V' (as
// V'(b, a), herm times it), at the rows' places, scattered over the column; without
// Hermiticity at its own place.
// Every element of V, U and V' is read or written once from HBM.  Both passes are products
// with small matrices and run on the FP64 matrix units; D is kept as their operand: the 64
// values of fragment (16 columns c, 4 rows k) of a group lie together, lane l's D(4k + l/16,
// 16c + l%16), zero past the group.  Bound by HBM: two passes of two-body size, read and
// written, 293 MB each at emax = 10.  There the first takes 178 us (368 with V and D staged
// in LDS and vector sums) and the second 269 us (700 with a row of V' per thread on four
// columns of T in LDS, its D column from the L2; 571 on the matrix units like that).
typedef double xfd4 __attribute__((ext_vector_type(4)));

// D blocks, one work-group per group g (the formula of k_hf_D).
__global__ __launch_bounds__(256) void k_xf_D(const BasisDev *bd, XformDev X, const double *C, double *Dg) {
  const BasisDev &B = *bd;
  const int g = blockIdx.x, s = X.g_start[g], m = X.g_start[g + 1] - s, ch = X.g_ch[g], J = ch / 6;
  const long N = B.norb;
  const int *kets = B.ch_kets + B.ch_kstart[ch];
  const int nks = (m + 3) >> 2, nel = 64 * nks * ((m + 15) >> 4);
  for (int e = threadIdx.x; e < nel; e += blockDim.x) {
    const int f = e >> 6, r = 4 * (f % nks) + ((e >> 4) & 3), c = 16 * (f / nks) + (e & 15);
    double d = 0.0;
    if (r < m && c < m) {
      const int ki = kets[X.g_kets[s + r]], ka = kets[X.g_kets[s + c]];
      const int p = B.kp[ki], q = B.kq[ki], pp = B.kp[ka], qq = B.kq[ka];
      d = C[p + pp * N] * C[q + qq * N];
      if (p != q) {
        const double ph = (((B.j2[p] + B.j2[q]) / 2 + 1 + J) & 1) ? -1.0 : 1.0;
        double x = C[q + pp * N] * C[p + qq * N];
        d += ph * x;
      }
      if (p == q) d *= 1.4142135623730951;
      if (pp == qq) d /= 1.4142135623730951;
    }
    Dg[X.g_doff[g] + e] = d;
  }
}

// One pass on one item (group g, rows r0 .. r0 + kXfRows - 1 of the input): D's fragments in
// LDS, 16 rows of the input's columns of the group per wave straight into the other operand.
template <bool SECOND>
__global__ __launch_bounds__(256) void k_xf_pass(const BasisDev *bd, XformDev X, const double *V, const double *Dg,
                                                 double *out, const int2 *items, double herm) {
  extern __shared__ __align__(16) double lds[];
  const BasisDev &B = *bd;
  const int2 it = items[blockIdx.x];
  if (it.x < 0) return;  // empty item (padding of an XCD run)
  const int g = it.x, r0 = it.y, s = X.g_start[g], m = X.g_start[g + 1] - s, ch = X.g_ch[g];
  const int n = B.ch_n[ch], nks = (m + 3) >> 2, nc = (m + 15) >> 4;
  const long off = B.ch_off[ch];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const double *Vc = V + off;
  double *oc = out + off;
  const int cs = X.g_start[X.c_start[ch]];  // the channel's first entry of g_kets
  int *ket = (int *)(lds + 64 * nks * nc);  // the group's kets, past it the last one
  for (int e = threadIdx.x; e < 16 * nc; e += blockDim.x) ket[e] = X.g_kets[s + min(e, m - 1)];
  for (int e = threadIdx.x; e < 64 * nks * nc; e += blockDim.x) lds[e] = Dg[X.g_doff[g] + e];
  __syncthreads();
  for (int rb = r0 + 16 * wv; rb < min(n, r0 + kXfRows); rb += 64) {
    const int row = rb + (lane & 15);
    const double *v = Vc + min(row, n - 1);
    double a[kXfMaxM / 4];
#pragma unroll
    for (int k = 0; k < kXfMaxM / 4; ++k)
      if (k < nks) a[k] = v[(long)ket[4 * k + (lane >> 4)] * n];
    const double f = herm != 0.0 ? herm : 1.0;
    const int to = SECOND ? X.g_kets[cs + min(row, n - 1)] : 0;  // the row's place in V'
    bool nan = false;
    for (int c = 0; c < nc; ++c) {
      xfd4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < kXfMaxM / 4; ++k)
        if (k < nks) {
          const double d = lds[(c * nks + k) * 64 + lane];
          acc = SECOND ? __builtin_amdgcn_mfma_f64_16x16x4f64(d, a[k], acc, 0, 0, 0)
                       : __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], d, acc, 0, 0, 0);
        }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (SECOND) {  // column 4 q + lane / 16, row lane % 16
          const int col = 16 * c + 4 * q + (lane >> 4);
          if (col < m && row < n) oc[herm != 0.0 ? (long)ket[col] * n + to : (long)to * n + ket[col]] = f * acc[q];
        } else {                 // row 4 q + lane / 16, column lane % 16
          const int col = 16 * c + (lane & 15), rr = rb + 4 * q + (lane >> 4);
          if (col < m && rr < n) oc[(long)rr * n + s - cs + col] = acc[q];
        }
      }
      if (c == 0) nan = __builtin_isnan((acc[0] + acc[1]) + (acc[2] + acc[3]));
    }
    // The last fragment repeats the group's last ket against zeros of D, which makes NaN of an
    // infinite one: such rows' results again, without them (the whole transformation at emax =
    // 10 525 -> 532 us; with 0 in its place among the loads 552 to 632).
    if ((m & 3) && __any(nan))
      for (int col = lane >> 4; col < m; col += 4) {
        double x = 0.0;
        for (int k = 0; k < m; ++k)
          x += v[(long)ket[k] * n] * lds[((col >> 4) * nks + (k >> 2)) * 64 + 16 * (k & 3) + (col & 15)];
        if (__builtin_isfinite(x) || row >= n) continue;
        if constexpr (SECOND)
          oc[herm != 0.0 ? (long)ket[col] * n + to : (long)to * n + ket[col]] = f * x;
        else
          oc[(long)row * n + s - cs + col] = x;
      }
  }
}

// One-body part, C^T O C with C block diagonal: out(a, b) = sum over k in a's block
// and l in b's block of C(k, a) O(k, l) C(l, b); one thread per element.
__global__ __launch_bounds__(256) void k_xf_one(const BasisDev *bd, const double *C, const double *O, double *out) {
  const BasisDev &B = *bd;
  const int N = B.norb;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= N * N) return;
  const int a = e % N, b = e / N;
  double acc = 0.0;
  for (int ik = B.obstart[a]; ik < B.obstart[a + 1]; ++ik) {
    const int k = B.oblist[ik];
    double t = 0.0;
    for (int il = B.obstart[b]; il < B.obstart[b + 1]; ++il) {
      const int l = B.oblist[il];
      t += O[k + (long)l * N] * C[l + (long)b * N];
    }
    acc += C[k + (long)a * N] * t;
  }
  out[e] = acc;
}

hipError_t launch_xform_blocks(const BasisDev *bd, const BasisDev &bh, const XformDev &X, const double *C,
                               const double *op, double *out, double *T, double *Dg, double *one_tmp,
                               const int2 *items, int nitems, int herm, hipStream_t s) {
  if (X.ngroups > 0) {
    hipLaunchKernelGGL(k_xf_D, dim3(X.ngroups), dim3(256), 0, s, bd, X, C, Dg);
    const size_t nc = (X.maxm + 15) / 16, lds = 512 * ((X.maxm + 3) / 4) * nc + 64 * nc;
    hipLaunchKernelGGL(k_xf_pass<false>, dim3(nitems), dim3(256), lds, s, bd, X, op + bh.two_off, Dg, T, items, 1.0);
    hipLaunchKernelGGL(k_xf_pass<true>, dim3(nitems), dim3(256), lds, s, bd, X, T, Dg, out + bh.two_off, items,
                       (double)herm);
  }
  const int n1 = bh.norb * bh.norb;
  if (n1 > 0) {
    hipLaunchKernelGGL(k_xf_one, dim3((n1 + 255) / 256), dim3(256), 0, s, bd, C, op + bh.one_off, one_tmp);
    hipError_t e = hipMemcpyAsync(out + bh.one_off, one_tmp, sizeof(double) * n1, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return e;
  }
  return hipGetLastError();
}

hipError_t launch_hf_D(const BasisDev *bd, const BasisDev &bh, const double *C, double *D, hipStream_t s) {
  if (bh.tbsize > 0) {
    const long nb = (bh.tbsize + 255) / 256;
    hipLaunchKernelGGL(k_hf_D, dim3((unsigned)nb), dim3(256), 0, s, bd, C, D);
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Counter-based N(0,1): SplitMix64 of (seed, index) -> two uniforms -> Box-Muller.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
__device__ __forceinline__ double normal_at(unsigned long long seed, unsigned long long idx) {
  unsigned long long a = splitmix64(seed ^ splitmix64(2 * idx + 1));
  unsigned long long b = splitmix64(a ^ 0x5851F42D4C957F2Dull);
  double u1 = ((a >> 11) + 1.0) * (1.0 / 9007199254740993.0);  // (0, 1]
  double u2 = (b >> 11) * (1.0 / 9007199254740992.0);          // [0, 1)
  return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

__global__ __launch_bounds__(256) void k_fill_random(const BasisDev *bd, double *op, int herm, unsigned long long seed) {
  const BasisDev &B = *bd;
  const double inv_sqrt2 = 0.7071067811865476;
  const long n2 = (long)B.norb * B.norb;
  const long total = n2 + B.tbsize;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    if (e < n2) {
      const int p = e % B.norb, q = e / B.norb;
      double v = 0.0;
      if (B.l[p] == B.l[q] && B.j2[p] == B.j2[q] && B.tz2[p] == B.tz2[q]) {
        // the value of the pair is formed once from the canonical (lo, hi) order,
        // so that (p,q) and (q,p) are exactly herm-related
        const int lo = min(p, q), hi = max(p, q);
        const int m = B.obstart[p + 1] - B.obstart[p];
        double a = normal_at(seed, (unsigned long long)((long)hi * B.norb + lo));
        double b = normal_at(seed, (unsigned long long)((long)lo * B.norb + hi));
        double vc = (lo == hi) ? (herm == 1 ? 2.0 * a : 0.0) : (a + herm * b);
        vc = vc * inv_sqrt2 / sqrt((double)m);
        v = (p <= q) ? vc : herm * vc;
      }
      op[B.one_off + e] = v;
    } else {
      const long t = e - n2;
      int clo = 0, chi = B.nch - 1;  // last channel starting at or before t (non-empty)
      while (clo < chi) {
        int mid = (clo + chi + 1) / 2;
        if (B.ch_off[mid] <= t) clo = mid; else chi = mid - 1;
      }
      const int ch = clo;
      const int n = B.ch_n[ch];
      const long loc = t - B.ch_off[ch];
      const int r = loc % n, c = loc / n;
      const int lo = min(r, c), hi = max(r, c);
      double a = normal_at(seed, (unsigned long long)(n2 + B.ch_off[ch] + (long)hi * n + lo));
      double b = normal_at(seed, (unsigned long long)(n2 + B.ch_off[ch] + (long)lo * n + hi));
      double vc = (lo == hi) ? (herm == 1 ? 2.0 * a : 0.0) : (a + herm * b);
      vc = vc * inv_sqrt2 / sqrt((double)n);
      op[B.two_off + t] = (r <= c) ? vc : herm * vc;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) op[0] = 0.0;
}

hipError_t launch_fill_random(const BasisDev *bd, const BasisDev &bh, double *op, int herm, unsigned long long seed,
                              hipStream_t s) {
  long total = (long)bh.norb * bh.norb + bh.tbsize;
  hipLaunchKernelGGL(k_fill_random, dim3(grid_for(total)), dim3(256), 0, s, bd, op, herm, seed);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// White generator, Epstein-Nesbet denominators (src/Generator.cc:110-188, 236-291).
__device__ double tbme_norm_u(const BasisDev &B, const double *two, int J, int a, int b, int c, int d) {
  int pab = (B.l[a] + B.l[b]) & 1, pcd = (B.l[c] + B.l[d]) & 1;
  if (pab != pcd) return 0.0;
  int tab = (B.tz2[a] + B.tz2[b]) / 2, tcd = (B.tz2[c] + B.tz2[d]) / 2;
  if (tab != tcd || J > B.jmax) return 0.0;
  int k1 = ket_index(B.norb, min(a, b), max(a, b)), k2 = ket_index(B.norb, min(c, d), max(c, d));
  int i = B.kmap[(long)k1 * (B.jmax + 1) + J], k = B.kmap[(long)k2 * (B.jmax + 1) + J];
  if (i < 0 || k < 0) return 0.0;
  int ch = 6 * J + 2 * (tab + 1) + pab;
  double ph = 1.0;
  if (a > b) ph *= sgn_parity((B.j2[a] + B.j2[b]) / 2 + 1 + J);
  if (c > d) ph *= sgn_parity((B.j2[c] + B.j2[d]) / 2 + 1 + J);
  return ph * two[B.ch_off[ch] + (long)k * B.ch_n[ch] + i];
}
__device__ double monopole_u(const BasisDev &B, const double *two, int a, int b, int c, int d) {
  double nrm = (a == b ? 1.4142135623730951 : 1.0) * (c == d ? 1.4142135623730951 : 1.0);
  int jmin = abs(B.j2[a] - B.j2[b]) / 2, jmax = (B.j2[a] + B.j2[b]) / 2;
  double mon = 0.0;
  for (int J = jmin; J <= jmax; ++J) mon += (2 * J + 1) * tbme_norm_u(B, two, J, a, b, c, d);
  mon /= (B.j2[a] + 1) * (B.j2[b] + 1);
  return nrm * mon;
}

// one-body part: one thread per (a core, i non-core)
__global__ __launch_bounds__(256) void k_white1(const BasisDev *bd, const double *H, double *Eta) {
  const BasisDev &B = *bd;
  const int norb = B.norb;
  const double *H1 = H + B.one_off, *H2 = H + B.two_off;
  double *E1 = Eta + B.one_off;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < (long)norb * norb;
       e += (long)gridDim.x * blockDim.x) {
    const int i = e % norb, a = e / norb;
    if (B.cvq[a] != 0 || B.cvq[i] == 0) continue;
    double d = H1[(long)i * norb + i] - H1[(long)a * norb + a];
    d += (B.occ[i] - B.occ[a]) * monopole_u(B, H2, i, a, i, a);
    if (fabs(d) < 1e-6) d = 1e-6;
    const double v = H1[(long)a * norb + i] / d;
    E1[(long)a * norb + i] = v;
    E1[(long)i * norb + a] = -v;
  }
}

// two-body part: block per channel, threads over (core ket, non-core ket)
__global__ __launch_bounds__(256) void k_white2(const BasisDev *bd, const double *H, double *Eta,
                                                const int4 *items) {
  const BasisDev &B = *bd;
  const int ch = items[blockIdx.x].y;
  const int n = B.ch_n[ch];
  const long off = B.ch_off[ch];
  const int norb = B.norb;
  const double *H1 = H + B.one_off, *H2 = H + B.two_off;
  double *E2 = Eta + B.two_off + off;
  const int c0 = B.gcore_start[ch], nc = B.gcore_start[ch + 1] - c0;
  const int q0 = B.gnc_start[ch], nq = B.gnc_start[ch + 1] - q0;
  const int ks = B.ch_kstart[ch];
  // eight lanes per element, six of them a monopole each: one after the other they are a
  // chain of loads six times as long
  const int lane = threadIdx.x & 63, m = lane & 7, first = lane & ~7;
  const int nt = nc * nq, step = gridDim.y * blockDim.x / 8;
  for (int t0 = (blockIdx.y * blockDim.x + threadIdx.x) / 8; t0 < (nt + 7) / 8 * 8; t0 += step) {  // whole waves
    const int t = min(t0, nt - 1);
    const int iket = B.gcore_loc[c0 + t / nq], ibra = B.gnc_loc[q0 + t % nq];
    const int kb = B.ch_kets[ks + ibra], kk = B.ch_kets[ks + iket];
    const int i = B.kp[kb], j = B.kq[kb], k = B.kp[kk], l = B.kq[kk];
    const double ni = B.occ[i], nj = B.occ[j], nk = B.occ[k], nl = B.occ[l];
    // (i, j), (k, l), (i, k), (i, l), (j, k), (j, l)
    const int p = m == 0 || m == 2 || m == 3 ? i : m == 1 ? k : j;
    const int q = m == 0 ? j : m == 1 || m == 3 || m == 5 ? l : k;
    const double mon = m < 6 ? monopole_u(B, H2, p, q, p, q) : 0.0;
    double d = H1[(long)i * norb + i] + H1[(long)j * norb + j] - H1[(long)k * norb + k] - H1[(long)l * norb + l];
    d += (1 - ni - nj) * __shfl(mon, first, 64);
    d -= (1 - nk - nl) * __shfl(mon, first + 1, 64);
    d += (ni - nk) * __shfl(mon, first + 2, 64);
    d += (ni - nl) * __shfl(mon, first + 3, 64);
    d += (nj - nk) * __shfl(mon, first + 4, 64);
    d += (nj - nl) * __shfl(mon, first + 5, 64);
    if (m != 0 || t0 >= nt) continue;
    if (fabs(d) < 1e-6) d = 1e-6;
    const double v = H2[off + (long)iket * n + ibra] / d;
    E2[(long)iket * n + ibra] = v;
    E2[(long)ibra * n + iket] = -v;
  }
}

hipError_t launch_white(const BasisDev *bd, const BasisDev &bh, const double *H, double *Eta, const int4 *gen_items,
                        int ngen, hipStream_t s) {
  long n2 = (long)bh.norb * bh.norb;
  hipLaunchKernelGGL(k_white1, dim3(grid_for(n2)), dim3(256), 0, s, bd, H, Eta);
  // 16 work-groups per channel: one took its elements in several turns (emax = 6: 54 us, 28 us
  // with eight, 20 with a lane per monopole)
  if (ngen > 0) hipLaunchKernelGGL(k_white2, dim3(ngen, 16), dim3(256), 0, s, bd, H, Eta, gen_items);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Whether two streams run at the same time: k_meet_wait on one stream waits at most
// `ticks` of the 100 MHz clock for the flag that k_meet_set raises on the other, and
// reports in met[1] whether it saw it.
__global__ void k_meet_wait(int *met, long long ticks) {
  const long long t0 = wall_clock64();
  int seen = 0;
  do {
    seen = __hip_atomic_load(met, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } while (!seen && wall_clock64() - t0 < ticks);
  met[1] = seen;
}
__global__ void k_meet_set(int *met) { __hip_atomic_store(met, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
hipError_t launch_meet(int *met, long long ticks, hipStream_t waiter, hipStream_t setter) {
  hipLaunchKernelGGL(k_meet_wait, dim3(1), dim3(1), 0, waiter, met, ticks);
  hipLaunchKernelGGL(k_meet_set, dim3(1), dim3(1), 0, setter, met);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
typedef double dbl4u __attribute__((ext_vector_type(4)));
// One wave: out[0..255] = D with A-operand = lane id, B-operand = 1;
//           out[256..511] = D with A-operand = 1, B-operand = lane id.
__global__ void k_mfma_probe(double *out) {
  const int lane = threadIdx.x;
  dbl4u z = {0.0, 0.0, 0.0, 0.0};
  dbl4u r1 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)lane, 1.0, z, 0, 0, 0);
  dbl4u r2 = __builtin_amdgcn_mfma_f64_16x16x4f64(1.0, (double)lane, z, 0, 0, 0);
  typedef float flt4u __attribute__((ext_vector_type(4)));
  flt4u zf = {0.f, 0.f, 0.f, 0.f};
  flt4u f1 = __builtin_amdgcn_mfma_f32_16x16x4f32((float)lane, 1.0f, zf, 0, 0, 0);
  flt4u f2 = __builtin_amdgcn_mfma_f32_16x16x4f32(1.0f, (float)lane, zf, 0, 0, 0);
  for (int q = 0; q < 4; ++q) {
    out[lane * 4 + q] = r1[q];
    out[256 + lane * 4 + q] = r2[q];
    out[512 + lane * 4 + q] = f1[q];
    out[768 + lane * 4 + q] = f2[q];
  }
}
hipError_t launch_mfma_probe(double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, s, out);
  return hipGetLastError();
}

// One v_mfma_f32_16x16x32_bf16 with lane l's operand slots j = 0..7 taken from
// a[8l + j], b[8l + j] (rounded to bf16) and C = 0; d[4l + q] = register q of
// lane l.  One wave, 512 + 512 inputs, 256 outputs.
__global__ void k_mfma_bf16_probe(const float *a, const float *b, float *d) {
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  typedef float flt4u __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x;
  bf16x8 va, vb;
  for (int j = 0; j < 8; ++j) {
    va[j] = (__bf16)a[lane * 8 + j];
    vb[j] = (__bf16)b[lane * 8 + j];
  }
  const flt4u z = {0.f, 0.f, 0.f, 0.f};
  const flt4u r = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, vb, z, 0, 0, 0);
  for (int q = 0; q < 4; ++q) d[lane * 4 + q] = r[q];
}
hipError_t launch_mfma_bf16_probe(const float *a, const float *b, float *d, hipStream_t s) {
  hipLaunchKernelGGL(k_mfma_bf16_probe, dim3(1), dim3(64), 0, s, a, b, d);
  return hipGetLastError();
}

}  // namespace imsrg
