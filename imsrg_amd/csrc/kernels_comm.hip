// kernels_comm.hip -- HIP kernels of the scalar IMSRG(2) commutator Z = [X, Y]
// on CDNA4 (gfx950).  Every kernel reads work items (int4: pair, a, b, c)
// so that one launch can cover all channels of one or many operator pairs.
//
// Two-body accumulation scheme: for Hermitian / anti-Hermitian Z every term
// adds only to the upper triangle (row <= col) of each channel block; the
// mirror kernel writes the lower triangle as hZ * upper at the end.  This is
// exact because each term of the reference produces a contribution whose
// (s,r) element is hZ times its (r,s) element (src/Commutator.cc:929, 1185-1194,
// 1611-1612).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "internal.hpp"
#include "launch.hpp"

namespace imsrg {

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

// Column (within a 16x16 block) held by register q of a lane in the D^T-block
// formulation of the GEMM kernels: f64 16x16x4 puts D[m][n] in lane n+16(m%4),
// register m/4; f32 16x16x4 in lane n+16(m/4), register m%4.
template <bool MIXED>
__device__ __forceinline__ int mfma_col(int lane, int q) {
  return MIXED ? 4 * (lane >> 4) + q : 4 * q + (lane >> 4);
}

#define SQRT2_D 1.4142135623730951

__device__ __forceinline__ double X1at(const double *one, int norb, int p, int q) { return one[(long)q * norb + p]; }

// Normalized scalar TBME <ab|V|cd>_J with the swapped-ket phases of
// TwoBodyME::GetTBME_norm (src/TwoBodyME.cc:128-147).
__device__ __forceinline__ double tbme_norm(const BasisDev &B, const double *two, int J, int a, int b, int c, int d) {
  int pab = (B.l[a] + B.l[b]) & 1, pcd = (B.l[c] + B.l[d]) & 1;
  if (pab != pcd) return 0.0;
  int tab = (B.tz2[a] + B.tz2[b]) / 2, tcd = (B.tz2[c] + B.tz2[d]) / 2;
  if (tab != tcd || J > B.jmax) return 0.0;
  int k1 = ket_index(B.norb, min(a, b), max(a, b));
  int k2 = ket_index(B.norb, min(c, d), max(c, d));
  int i = B.kmap[(long)k1 * (B.jmax + 1) + J];
  int k = B.kmap[(long)k2 * (B.jmax + 1) + J];
  if (i < 0 || k < 0) return 0.0;
  int ch = 6 * J + 2 * (tab + 1) + pab;
  double ph = 1.0;
  if (a > b) ph *= sgn_parity((B.j2[a] + B.j2[b]) / 2 + 1 + J);
  if (c > d) ph *= sgn_parity((B.j2[c] + B.j2[d]) / 2 + 1 + J);
  return ph * two[B.ch_off[ch] + (long)k * B.ch_n[ch] + i];
}

template <int NV>
__device__ __forceinline__ void block_reduce(double (&v)[NV]) {
  __shared__ double red[NV][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double x = v[q];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_down(x, o, 64);
    if (lane == 0) red[q][w] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = (red[q][0] + red[q][1]) + (red[q][2] + red[q][3]);
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// comm110ss (src/Commutator.cc:564-581) and comm220ss (601-631) -> Z0.
// Block 0 of a pair clears Z's one-body block and forms the comm110 sum, block
// 1+ch the comm220 contribution of channel ch; partial sums go to scratch and
// final_zero adds them in channel order.
__device__ __forceinline__ void front_zero(const PairPtrs &P, int bid) {
  const BasisDev &B = *P.basis;
  const int norb = B.norb;
  if (bid > B.nch) return;
  double acc[1] = {0.0};
  const bool skip = (P.hX == P.hY);
  if (bid == 0) {
    const double *X1 = P.X + B.one_off, *Y1 = P.Y + B.one_off;
    double *Z1 = P.Z + B.one_off;
    for (int e = threadIdx.x; e < norb * norb; e += blockDim.x) Z1[e] = 0.0;
    if (!skip && (P.mask & M110)) {
      for (int t = threadIdx.x; t < B.nholes * norb; t += blockDim.x) {
        int a = B.holes[t / norb], k = t % norb;
        double xy = X1at(X1, norb, a, k) * X1at(Y1, norb, k, a);
        double yx = X1at(Y1, norb, a, k) * X1at(X1, norb, k, a);
        acc[0] += (B.j2[a] + 1) * B.occ[a] * (xy - yx);
      }
    }
  } else if (!skip && (P.mask & M220)) {
    const int ch = bid - 1;
    const int h0 = B.hh_start[ch], nhh = B.hh_start[ch + 1] - h0;
    if (nhh > 0) {
      const int n = B.ch_n[ch];
      const long off = B.ch_off[ch];
      const double *X2 = P.X + B.two_off + off, *Y2 = P.Y + B.two_off + off;
      const double *w = B.w220 + B.ch_kstart[ch];
      const double f = 2.0 * (2 * (ch / 6) + 1);
      // X(h,m) = hX X(m,h): both operands read down column h
      for (int t = threadIdx.x; t < nhh * n; t += blockDim.x) {
        int ih = t / n, m = t % n;
        int h = B.hh_loc[h0 + ih];
        acc[0] += f * B.hh_occ[h0 + ih] * ((P.hX * X2[(long)h * n + m]) * (Y2[(long)h * n + m] * w[m]));
      }
    }
  }
  block_reduce<1>(acc);
  if (threadIdx.x == 0) P.scratch[bid] = acc[0];
}

// Z0 from the partial sums: one work-group per pair, the channels' sums staged in
// LDS (`buf`, nbuf doubles) and added in channel order by one thread.
__device__ __forceinline__ void final_zero(const PairPtrs &P, double *buf, int nbuf) {
  const int nch = P.basis->nch;
  double s220 = 0.0;
  for (int c0 = 0; c0 < nch; c0 += nbuf) {
    const int m = min(nbuf, nch - c0);
    for (int c = threadIdx.x; c < m; c += blockDim.x) buf[c] = P.scratch[1 + c0 + c];
    __syncthreads();
    if (threadIdx.x == 0)
      for (int c = 0; c < m; ++c) s220 += buf[c];
    __syncthreads();
  }
  if (threadIdx.x == 0) P.Z[0] = (0.0 + P.scratch[0]) + s220;
}

// ---------------------------------------------------------------------------
// One-body terms for one (i, j) pair of the same (l, j2, tz2) block, i <= j:
// comm111ss (src/Commutator.cc:644-649), comm121ss (670-728) and the one-body
// part of comm222_pp_hh_221ss (1246-1294).  M_pp / M_hh elements are formed
// directly as folded dot products, M(r,s) + hZ M(s,r) with M = X W Y.
__device__ __forceinline__ double fold_dot(const double *xr, const double *xs, const double *yr, const double *ys,
                                           const int *loc, const double *w, int nk, int start, int stride,
                                           double hZ) {
  // the two products summed apart, as the reference's M and its transpose: for
  // r == s and hZ = -1 they cancel exactly (an anti-Hermitian diagonal is 0)
  double m1 = 0.0, m2 = 0.0;
  for (int q = start; q < nk; q += stride) {
    const int k = loc[q];
    m1 += w[q] * (xr[k] * ys[k]);
    m2 += w[q] * (xs[k] * yr[k]);
  }
  return m1 + hZ * m2;
}

__device__ __forceinline__ void front_one(const PairPtrs &P, const int4 &it) {
  const BasisDev &B = *P.basis;
  const int norb = B.norb, i = it.y, j = it.z;
  const double *X1 = P.X + B.one_off, *Y1 = P.Y + B.one_off;
  const double *X2 = P.X + B.two_off, *Y2 = P.Y + B.two_off;
  // (X1 Y1)(i,j) and (Y1 X1)(i,j) summed apart, as the reference's two matrix
  // products: commuting blocks then give exactly 0
  double acc[3] = {0.0, 0.0, 0.0};
  if (P.mask & M111) {
    for (int k = threadIdx.x; k < norb; k += blockDim.x) {
      acc[0] += X1at(X1, norb, i, k) * X1at(Y1, norb, k, j);
      acc[2] += X1at(Y1, norb, i, k) * X1at(X1, norb, k, j);
    }
  }
  if (P.mask & M121) {
    // one task per (hole a, partner b, monopole term, J): the monopoles'
    // (2J+1)-weighted elements spread over the lanes, so that a lane waits for one
    // chain of index loads in place of one per J
    const int nJ = B.j2[i] + 1;  // at most this many J couple an orbit with i
    const int ntask = B.nholes * B.maxblk * 4 * nJ;
    for (int t = threadIdx.x; t < ntask; t += blockDim.x) {
      const int dJ = t % nJ, u = t / nJ;
      const int term = u & 3, ib = (u >> 2) % B.maxblk, ia = (u >> 2) / B.maxblk;
      const int a = B.holes[ia];
      const int o0 = B.obstart[a];
      if (ib >= B.obstart[a + 1] - o0) continue;
      const int b = B.oblist[o0 + ib];  // j_b = j_a
      const double nanb = B.occ[a] * (1.0 - B.occ[b]);
      if (fabs(nanb) < 1e-6) continue;
      const int ja = B.j2[a], ji = B.j2[i], J = abs(ja - ji) / 2 + dJ;
      if (J > (ja + ji) / 2) continue;
      const int x = (term & 1) ? a : b, y = (term & 1) ? b : a;  // <x i | y j>
      double v = (2 * J + 1) * tbme_norm(B, term < 2 ? Y2 : X2, J, x, i, y, j);
      v *= (x == i ? SQRT2_D : 1.0) * (y == j ? SQRT2_D : 1.0);
      v *= nanb * ((term & 1) ? X1at(term < 2 ? X1 : Y1, norb, b, a) : X1at(term < 2 ? X1 : Y1, norb, a, b));
      // (2 j_a + 1) over the monopole's (2 j_a + 1)(2 j_i + 1)
      acc[1] += ((term == 1 || term == 2) ? -v : v) / (ji + 1);
    }
  }
  block_reduce<3>(acc);
  if (threadIdx.x == 0) P.obpart[B.ob_start[it.w]] = (acc[0] - acc[2]) + acc[1];
}

// Lane's share of (2J+1) fac M(ci, cj) for the comm221 one-body part
// (src/Commutator.cc:1246-1294): M = M_pp (pp = true, ConstructScalarMpp_Mhh's
// pp list) or M_hh, formed as the folded dot product M(r,s) + hZ M(s,r) over
// the list entries start, start + stride, ...; 0 when a ket is missing.
__device__ __forceinline__ double m221_part(const BasisDev &B, const double *X2, const double *Y2, int i, int j,
                                            int c, int J, bool pp, int start, int stride, double hZ) {
  const int norb = B.norb, nJ = B.jmax + 1;
  const int kci = ket_index(norb, min(c, i), max(c, i)), kcj = ket_index(norb, min(c, j), max(c, j));
  const int r = B.kmap[(long)kci * nJ + J], s = B.kmap[(long)kcj * nJ + J];
  if (r < 0 || s < 0) return 0.0;
  const int ch = 6 * J + 2 * ((B.tz2[c] + B.tz2[i]) / 2 + 1) + ((B.l[c] + B.l[i]) & 1);
  const int n = B.ch_n[ch];
  const long off = B.ch_off[ch];
  double fac = (c == i ? SQRT2_D : 1.0) * (c == j ? SQRT2_D : 1.0);
  if (c > i) fac *= sgn_parity((B.j2[c] + B.j2[i]) / 2 + 1 + J);
  if (c > j) fac *= sgn_parity((B.j2[c] + B.j2[j]) / 2 + 1 + J);
  const double *xr = X2 + off + (long)r * n, *xs = X2 + off + (long)s * n;
  const double *yr = Y2 + off + (long)r * n, *ys = Y2 + off + (long)s * n;
  const int k0 = pp ? B.kpp_start[ch] : B.khh_start[ch], k1 = pp ? B.kpp_start[ch + 1] : B.khh_start[ch + 1];
  const double m = pp ? fold_dot(xr, xs, yr, ys, B.kpp_loc + k0, B.kpp_w + k0, k1 - k0, start, stride, hZ)
                      : fold_dot(xr, xs, yr, ys, B.khh_loc + k0, B.khh_w + k0, k1 - k0, start, stride, hZ);
  return (2 * J + 1) * fac * m;
}

// comm221 one-body part in partial sums, one slot per item (it.w):
//  kind 0 (n_c != 0): n_c M_pp for 4 entries (c, J) of the list ob_cj (one per wave), the
//  wave's lanes over the pp list;
//  kind 1 (1 - n_c != 0): (1 - n_c) M_hh for 16 orbits c of the list cpart, 16 lanes on
//  each, over J and the hh lists.
// A work-group is a chain of index loads with little work behind it: kind 0 by the block
// and kind 1 by the wave, with four times the work-groups, took 481 us in a batch of 48
// pairs at emax 4-7 with the other work-groups before the Pandya chunks (now 232), and the
// first launch 68 us at emax = 8 (58) and 550 at emax = 12 (505).
__device__ __forceinline__ void front_221(const PairPtrs &P, const int4 &it) {
  const BasisDev &B = *P.basis;
  const int2 pr = B.pairs1[it.y];
  const int i = pr.x, j = pr.y;
  const double *X2 = P.X + B.two_off, *Y2 = P.Y + B.two_off;
  const double hZ = P.hZ;
  const int lane = threadIdx.x & 63;
  double acc[1] = {0.0};
  if (!(it.z >> 30)) {
    const int e = threadIdx.x >> 6;
    if (e <= (it.z >> 28 & 3)) {
      const int cj = B.ob_cj[(it.z & 0xfffffff) + e], c = cj >> 8, J = cj & 0xff;
      acc[0] = B.occ[c] * m221_part(B, X2, Y2, i, j, c, J, true, lane, 64, hZ);
    }
  } else {
    const int q = (it.z & 0x3fffffff) + (threadIdx.x >> 4);
    if (q < B.ncpart) {
      const int c = B.cpart[q];
      const int Jmin = max(abs(B.j2[c] - B.j2[i]), abs(B.j2[c] - B.j2[j])) / 2;
      const int Jmax = (B.j2[c] + min(B.j2[i], B.j2[j])) / 2;
      double m = 0.0;
      // eight J at a time, two lanes on each one's hh list (a few kets)
      for (int J = Jmin + (lane >> 1 & 7); J <= Jmax; J += 8) m += m221_part(B, X2, Y2, i, j, c, J, false, lane & 1, 2, hZ);
      acc[0] = (1.0 - B.occ[c]) * m;
    }
  }
  block_reduce<1>(acc);
  if (threadIdx.x == 0) P.obpart[it.w] = P.hX * acc[0];
}

// Z1(i, j) = comm111 + comm121 + comm221 / (j_i + 1) from the partial sums of
// one-body pair p, one wave per pair (lane-strided sums and a fixed shuffle
// tree: the same order every call), and Z1(j, i) = hZ Z1(i, j).
__device__ __forceinline__ void final_one(const PairPtrs &P, int blk) {
  const BasisDev &B = *P.basis;
  const int p = blk * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (p >= B.n1pairs) return;  // wave-uniform
  const int2 pr = B.pairs1[p];
  const int i = pr.x, j = pr.y, s0 = B.ob_start[p], s1 = B.ob_start[p + 1];
  double z221 = 0.0;
  if (P.mask & M221)
    for (int s = s0 + 1 + lane; s < s1; s += 64) z221 += P.obpart[s];
  for (int o = 32; o > 0; o >>= 1) z221 += __shfl_down(z221, o, 64);
  if (lane != 0) return;
  const double z = P.obpart[s0] + z221 / (B.j2[i] + 1.0);
  double *Z1 = P.Z + B.one_off;
  Z1[(long)j * B.norb + i] = z;
  if (i != j) Z1[(long)i * B.norb + j] = P.hZ * z;
}

// ---------------------------------------------------------------------------
// SYR2K tile on MFMA f64 16x16x4:
//   D(r,s) = alpha * cph(s) * sum_k w_k [ A(r,ka_k) B(s,kb_k) + h B(r,kb_k) A(s,ka_k) ],  r <= s
// with A, B column-major n x * matrices (A(r,k) = A[k*n + r]).
// MODE 0: pp/hh term of comm222_pp_hh_221ss (src/Commutator.cc:1171-1194, 1237-1238):
//         A = X2, B = Y2 of one channel, k over pp/hh kets with weight w_pp - w_hh,
//         alpha = hY, h = hZ.  (X W Y + hZ (X W Y)^T written with Y^T = hY Y.)
// MODE 1: head of Zbar in comm222_phss (src/Commutator.cc:1789-1799): A = Xbar,
//         B = Ybar^T, h = +1 (Z Hermitian) or -1.
// MODE 2: tail of Zbar (src/Commutator.cc:1788-1789, 1805): B columns permuted
//         by ab <-> ba with weights hY*phi(ph ket), cph(s) = phi(s), h = +1.
//
// MIXED: operands rounded to FP32 in LDS, products on f32 16x16x4 MFMA, FP32
// partial sums over kF32Flush k-steps added into the FP64 accumulators.
template <int MODE, bool MIXED>
__device__ __forceinline__ void syr2k_tile(const PairArg &pa, const int4 &it) {
  constexpr int LD = kTile + 2;
  using ST = typename std::conditional<MIXED, float, double>::type;
  // the FP32-product ph GEMM keeps Zbar in FP32 (its inverse Pandya gather reads
  // 4-byte elements); the FP64 kernels keep it in FP64
  using ZT = typename std::conditional<MIXED && MODE != 0, float, double>::type;
  __shared__ ST As[2][kTileK][LD];
  __shared__ ST Bs[2][kTileK][LD];
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const double *Am, *Bm;
  int n, nk, nph = 0;
  const int *kl = nullptr;
  const double *kw = nullptr;
  const int *phl = nullptr;
  const signed char *phi = nullptr;
  double alpha, h;
  double *D = nullptr;
  ZT *Dz = nullptr;
  if (MODE == 0) {
    const int ch = it.y;
    n = B.ch_n[ch];
    const long off = B.ch_off[ch];
    Am = P.X + B.two_off + off;
    Bm = P.Y + B.two_off + off;
    const int k0 = B.k_start[ch];
    nk = B.k_start[ch + 1] - k0;
    kl = B.k_loc + k0;
    kw = B.k_w + k0;
    alpha = (double)P.hY;
    h = (double)P.hZ;
    D = P.Z + B.two_off + off;
  } else {
    const int cc = it.y;
    n = B.cc_n[cc];
    nph = B.cc_nph[cc];
    nk = 2 * nph;
    const long xo = B.cc_xoff[cc];
    Am = P.Xt + xo;
    Bm = P.Yt + xo;
    Dz = reinterpret_cast<ZT *>(P.Zbar) + B.cc_zoff[cc] + (MODE == 2 ? (long)n * n : 0);
    alpha = 1.0;
    h = (MODE == 1) ? (P.hZ == 1 ? 1.0 : -1.0) : 1.0;
    phi = B.cc_phi + B.cc_kstart[cc];
    phl = B.cc_ph + B.cc_phstart[cc];
  }
  const int R0 = it.z * kTile, S0 = it.w * kTile;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = (wv & 1) * 32, wc = (wv >> 1) * 32;
  // 16x16 blocks with upper-triangle elements inside the matrix (the others issue no MFMA)
  unsigned bm = 0;
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      const int r0 = R0 + wr + mi * 16, c0 = S0 + wc + ni * 16;
      if (r0 < n && c0 < n && r0 <= c0 + 15) bm |= 1u << (mi * 2 + ni);
    }
  dbl4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = dbl4{0.0, 0.0, 0.0, 0.0};

  const int tk = threadIdx.x >> 4, tr = (threadIdx.x & 15) * 4;
  const int K2 = 2 * nk;
  // global -> register loads of one k-stage (16 values of k' per stage)
  auto load_stage = [&](int k0, double (&av)[4], double (&bv)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) av[q] = bv[q] = 0.0;
    const int kk = k0 + tk;
    if (kk < K2) {
      const int k = kk < nk ? kk : kk - nk;
      int ca, cb;
      double wk;
      if (MODE == 0) {
        ca = cb = kl[k];
        wk = kw[k];
      } else if (MODE == 1) {
        ca = cb = k;
        wk = 1.0;
      } else {
        ca = k;
        cb = k < nph ? k + nph : k - nph;
        wk = (double)P.hY * (double)phi[phl[k < nph ? k : k - nph]];
      }
      const double *sa, *sb;
      double fa;
      if (kk < nk) {
        sa = Am + (long)ca * n;
        sb = Bm + (long)cb * n;
        fa = wk;
      } else {
        sa = Bm + (long)cb * n;
        sb = Am + (long)ca * n;
        fa = wk * h;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = R0 + tr + q, c = S0 + tr + q;
        av[q] = (r < n) ? sa[r] * fa : 0.0;
        bv[q] = (c < n) ? sb[c] : 0.0;
      }
    }
  };
  double av[4], bv[4];
  load_stage(0, av, bv);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    As[0][tk][tr + q] = av[q];
    Bs[0][tk][tr + q] = bv[q];
  }
  __syncthreads();
  int cur = 0;
  for (int k0 = 0; k0 < K2; k0 += kTileK) {
    const bool more = k0 + kTileK < K2;
    if (more) load_stage(k0 + kTileK, av, bv);  // in flight during the MFMAs below
    if constexpr (MIXED) {
      flt4 t[2][2];
#pragma unroll
      for (int ks = 0; ks < kTileK / 4; ++ks) {
        const int kr = ks * 4 + (lane >> 4);
        const float a0 = As[cur][kr][wr + (lane & 15)], a1 = As[cur][kr][wr + 16 + (lane & 15)];
        const float b0 = Bs[cur][kr][wc + (lane & 15)], b1 = Bs[cur][kr][wc + 16 + (lane & 15)];
        const bool fresh = ks % kF32Flush == 0;
        const flt4 fz = {0.f, 0.f, 0.f, 0.f};
        if (bm & 1) t[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(b0, a0, fresh ? fz : t[0][0], 0, 0, 0);
        if (bm & 2) t[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b1, a0, fresh ? fz : t[0][1], 0, 0, 0);
        if (bm & 4) t[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(b0, a1, fresh ? fz : t[1][0], 0, 0, 0);
        if (bm & 8) t[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b1, a1, fresh ? fz : t[1][1], 0, 0, 0);
        if (ks % kF32Flush == kF32Flush - 1) {
#pragma unroll
          for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
              for (int q = 0; q < 4; ++q) acc[mi][ni][q] += (double)t[mi][ni][q];
        }
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < kTileK / 4; ++ks) {
        const int kr = ks * 4 + (lane >> 4);
        const double a0 = As[cur][kr][wr + (lane & 15)], a1 = As[cur][kr][wr + 16 + (lane & 15)];
        const double b0 = Bs[cur][kr][wc + (lane & 15)], b1 = Bs[cur][kr][wc + 16 + (lane & 15)];
        // D^T blocks: lane l, register q holds D row (lane&15), column mfma_col(l, q)
        if (bm & 1) acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, a0, acc[0][0], 0, 0, 0);
        if (bm & 2) acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, a0, acc[0][1], 0, 0, 0);
        if (bm & 4) acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, a1, acc[1][0], 0, 0, 0);
        if (bm & 8) acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, a1, acc[1][1], 0, 0, 0);
      }
    }
    if (more) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        As[cur ^ 1][tk][tr + q] = av[q];
        Bs[cur ^ 1][tk][tr + q] = bv[q];
      }
    }
    __syncthreads();
    cur ^= 1;
  }
  if (MODE == 0) {
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = R0 + wr + mi * 16 + (lane & 15);
          const int col = S0 + wc + ni * 16 + mfma_col<MIXED>(lane, q);
          if (row < n && col < n && row <= col) {
            const double v = alpha * acc[mi][ni][q];
            double *dp = D + (long)col * n + row;
            *dp = v;
          }
        }
  } else {
    // Zbar blocks are stored in full: the upper triangle as computed, the lower
    // one as (head) hZ-sign or (tail) phi_r phi_s times the upper element, as
    // the reference's folds make them (src/Commutator.cc:1792-1805).
    __shared__ double Tt[kTile][kTile + 1];
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int rr = wr + mi * 16 + (lane & 15), cc = wc + ni * 16 + mfma_col<MIXED>(lane, q);
          double v = alpha * acc[mi][ni][q];
          if (MODE == 2) {
            const int col = S0 + cc;
            v *= (col < n) ? (double)phi[col] : 0.0;
          }
          Tt[rr][cc] = v;
        }
    __syncthreads();
    for (int e = threadIdx.x; e < kTile * kTile; e += blockDim.x) {
      const int rr = e & (kTile - 1), cc = e / kTile;
      const int row = R0 + rr, col = S0 + cc;
      if (row < n && col < n && row <= col) Dz[(long)col * n + row] = (ZT)Tt[rr][cc];
      // mirrored element (S0+rr, R0+cc) from the upper element (R0+cc, S0+rr)
      const int row2 = S0 + rr, col2 = R0 + cc;
      if (row2 < n && col2 < n && row2 > col2) {
        const double sym = (MODE == 1) ? h : (double)(phi[row2] * phi[col2]);
        Dz[(long)col2 * n + row2] = (ZT)(sym * Tt[cc][rr]);
      }
    }
  }
}
template <int MODE, bool MIXED>
__global__ __launch_bounds__(256) void k_syr2k(PairArg pa, const int4 *items) {
  syr2k_tile<MODE, MIXED>(pa, items[blockIdx.x]);
}


// ---------------------------------------------------------------------------
// SYR2K on 128x128 output tiles: each of the 8 waves owns a 64x32 sub-tile
// (4x2 MFMA blocks), so one LDS read feeds two or four MFMAs; k-stages of 16 are
// double-buffered in LDS and filled by direct global->LDS copies issued one
// stage ahead.
//   D(r,s) = alpha * cph(s) * sum_k w_k [ A(r,ka_k) B(s,kb_k) + h B(r,kb_k) A(s,ka_k) ],  r <= s
// PH false: pp/hh term of comm222_pp_hh_221ss (src/Commutator.cc:1171-1194, 1237-1238):
//         A = X2, B = Y2 of one channel, k over pp/hh kets with weight w_pp - w_hh,
//         alpha = hY, h = hZ; the upper triangle of Z2 is written.
// PH true, head of Zbar in comm222_phss (src/Commutator.cc:1789-1799): A = Xbar,
//         B = Ybar^T, h = +1 (Z Hermitian) or -1.
// PH true, tail of Zbar (src/Commutator.cc:1788-1789, 1805): B columns permuted
//         by ab <-> ba with weights hY*phi(ph ket), cph(s) = phi(s), h = +1.
// The ph GEMM stores the upper triangle of Zbar and, of the lower one, the elements whose
// two kets have the same first orbit (all that the inverse Pandya reads): they lie within
// cc_run of the diagonal, so that sub-tiles further off leave their mirror image out.  The
// lower elements are (head) hZ-sign or (tail) phi_r phi_s times the upper ones, as the
// reference's folds make them (src/Commutator.cc:1792-1805).  Without the others the ph
// GEMM took 420 us at emax = 10 (FP64; 472 with them) and 335 us with FP32 products (355).
// MIXED (pp/hh, or with SPLIT; the ph GEMM with FP32 products is k_ph_big_f32): operands
// rounded to FP32 when read from LDS, products on f32 16x16x4 MFMA, FP32 partial sums
// over two stages (32 k) added into the FP64 accumulators.
// SPLIT (with MIXED): each operand is split into two FP32 values, a = ah + al
// with ah = fl32(a), al = fl32(a - ah), and a product takes three f32 MFMAs,
// ah*bh + ah*bl + al*bh (the dropped al*bl is 2^-48 of it); the FP32 partial
// sums are flushed into FP64 after every 4 k.
// Non-temporal stores: the last kernel's of Z, which is read again only by a later call.
__device__ __forceinline__ void st_nt(double *p, double v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void st_nt2(double *p, double a, double b) {
  typedef double d2v __attribute__((ext_vector_type(2)));
  const d2v v = {a, b};
  __builtin_nontemporal_store(v, reinterpret_cast<d2v *>(p));
}

// A wave of a 128x128 tile owns the 64 x kGW sub-tile at rows (w & 1) * 64,
// columns (w >> 1) * kGW; it has work when that sub-tile holds an upper-
// triangle element inside the n x n matrix.
__device__ __forceinline__ bool tile_wave_live(int R0, int S0, int n, int w) {
  return R0 + (w & 1) * 64 < n && S0 + (w >> 1) * kGW < n && R0 + (w & 1) * 64 <= S0 + (w >> 1) * kGW + kGW - 1;
}

// Stores a wave's sub-tile of a 128x128 tile from its FP64 accumulators (lane layout of the
// f32 MFMAs when F32L, else of the f64 16x16x4 MFMA): 16 consecutive rows of four columns
// per store instruction.
// PH false: the upper triangle of D = alpha * acc.
// PH true: Zbar, the upper triangle and the elements next to the diagonal in the lower one
// (less than run from it); s_ph holds the tile's row (0) and column (1) phases in the
// tail (h = 1) and 1 in the head.
// The elements used to go through LDS (the lower triangle was stored in full, transposed
// there) and to memory by non-temporal stores.  Stored at once, the waves wait for no other,
// and plain stores, whose lines the L2 completes from two instructions, are the faster ones
// here: ph GEMM at emax = 10 FP64 420 -> 395 us (435 with non-temporal stores), emax = 7 61 -> 56.
template <bool PH, bool F32L>
__device__ __forceinline__ void gemm_epilogue(const dbl4 (&acc)[4][kGN], double *D, int n, int R0, int S0,
                                              double alpha, double h, int run, const signed char (*s_ph)[kTileB]) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = (wv & 1) * 64, wc = (wv >> 1) * kGW;
  const bool near = PH && S0 + wc - (R0 + wr + 63) < run;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < kGN; ++ni)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int rr = wr + mi * 16 + (lane & 15), cc = wc + ni * 16 + mfma_col<F32L>(lane, q);
        const int row = R0 + rr, col = S0 + cc;
        if (row >= n || col >= n || row > col) continue;
        if constexpr (!PH) {
          D[(long)col * n + row] = alpha * acc[mi][ni][q];
        } else {
          const double v = acc[mi][ni][q] * (double)s_ph[1][cc];
          D[(long)col * n + row] = v;
          // the lower element: h phi_r phi_c times the upper one
          if (near && col != row && col - row < run)
            D[(long)row * n + col] = h * (double)(s_ph[1][cc] * s_ph[0][rr]) * v;
        }
      }
}

// The work-group's tile of a ph item list whose items are each done twice, head and
// tail, in one launch: runs of 8 work-groups (one per XCD) alternate between the two
// halves, so that an item's halves, which read the same panels, run close together on
// one XCD.  Small bases have fewer tiles than CUs and each tile is a chain of k-stages,
// so two launches one after the other took twice as long (emax = 5 FP32 53 -> 30 us,
// emax = 7 FP64 85 -> 61 us); emax = 10 517 -> 472 us FP64, 390 -> 357 us FP32.
__device__ __forceinline__ int4 ph_item(const int4 *items, int nitems, bool &tail) {
  const int i = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
  tail = (blockIdx.x >> 3) & 1;
  return i < nitems ? items[i] : make_int4(0, -1, 0, 0);
}

template <bool PH, bool MIXED, bool SPLIT = false>
__device__ __forceinline__ void gemm_tile(PairArg pa, const int4 *items, int nitems) {
  static_assert(MIXED || !SPLIT, "split products are a mixed-precision mode");
  constexpr int T = kTileB, LD = kTileB + 4;
  // operands stay FP64 in LDS (they arrive by direct global->LDS copies); the
  // mixed kernel rounds them to FP32 when it reads them
  // the two stage buffers are separate LDS objects and every access names one
  // statically (the stage loop is unrolled by two), so the compiler can tell
  // the reads of one buffer from the direct copies into the other and does
  // not wait for the copies in flight before computing
  __shared__ __align__(16) double A0[kTileK][LD], A1[kTileK][LD];
  __shared__ __align__(16) double B0[kTileK][LD], B1[kTileK][LD];
  __shared__ double W0[kTileK], W1[kTileK];
  bool tail = false;
  const int4 it = PH ? ph_item(items, nitems, tail) : items[blockIdx.x];
  if (it.y < 0) return;  // padding item of the XCD-balanced order
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  int n, nk, nph = 0;
  const double *Am, *Bm;
  const int *kl = nullptr;
  const double *kw = nullptr;
  const signed char *phi = nullptr, *phph = nullptr;
  double alpha, h;
  static_assert(!PH || MIXED == SPLIT, "the ph GEMM with FP32 products is k_ph_big_f32");
  double *D;
  if constexpr (!PH) {
    const int ch = it.y;
    n = B.ch_n[ch];
    const long off = B.ch_off[ch];
    Am = P.X + B.two_off + off;
    Bm = P.Y + B.two_off + off;
    const int k0s = B.k_start[ch];
    nk = B.k_start[ch + 1] - k0s;
    kl = B.k_loc + k0s;
    kw = B.k_w + k0s;
    alpha = (double)P.hY;
    h = (double)P.hZ;
    D = P.Z + B.two_off + off;
  } else {
    const int cc = it.y;
    n = B.cc_n[cc];
    nph = B.cc_nph[cc];
    nk = 2 * nph;
    const long xo = B.cc_xoff[cc];
    Am = P.Xt + xo;
    Bm = P.Yt + xo;
    D = P.Zbar + B.cc_zoff[cc] + (tail ? (long)n * n : 0);
    alpha = 1.0;
    h = tail || P.hZ == 1 ? 1.0 : -1.0;
    phi = B.cc_phi + B.cc_kstart[cc];
    phph = B.cc_phph + B.cc_phstart[cc];
  }
  const int R0 = it.z * T, S0 = it.w * T;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // ph: the phases of the tile's 128 rows and 128 columns (tail; 1 in the head), staged
  // once for the epilogue (the prologue's barrier below publishes them)
  __shared__ signed char s_ph[2][T];
  if constexpr (PH) {
    if (threadIdx.x < 2 * T) {
      const int sd = threadIdx.x / T, e = threadIdx.x - sd * T;
      s_ph[sd][e] = tail ? phi[min((sd ? S0 : R0) + e, n - 1)] : 1;
    }
  }
  // 8 waves, each a 64x32 sub-tile: rows wr .. wr+63, columns wc .. wc+31
  const int wr = (wv & 1) * 64, wc = (wv >> 1) * kGW;
  // a wave whose sub-tile holds no upper-triangle element inside the matrix
  // (padding past n, or below the diagonal) issues no MFMA
  const bool wave_live = tile_wave_live(R0, S0, n, wv);
  dbl4 acc[4][kGN];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < kGN; ++b) acc[a][b] = dbl4{0.0, 0.0, 0.0, 0.0};
  const int K2 = 2 * nk;
  // Stage loader: wave w copies the k' columns 2w, 2w+1 of the stage, for
  // the A and the B row block, each a 128-row segment of one column, with one
  // 16-byte-per-lane global->LDS copy (lane l: rows 2l, 2l+1).  Rows past n
  // are never written back; their source is clamped so that a row pair reads
  // at most one element past the column (inside the arena, or the buffer's
  // slack).  Column indices (wave-uniform) are loaded one stage ahead.
  const int ra = min(R0 + 2 * lane, n - 1), rb = min(S0 + 2 * lane, n - 1);
  // pp/hh: the channel's column-index list kl[0..nk) is staged in LDS (dynamic
  // shared memory of at least nk ints), so index reads never wait behind the
  // global->LDS copies in flight
  extern __shared__ int KLs[];
  if constexpr (!PH) {
    for (int e = threadIdx.x; e < nk; e += blockDim.x) KLs[e] = kl[e];
    __syncthreads();
  }
  auto load_idx = [&](int k0, int (&ki)[kGC]) {
#pragma unroll
    for (int j = 0; j < kGC; ++j) {
      const int kk = min(k0 + wv * kGC + j, K2 - 1);
      const int k = kk < nk ? kk : kk - nk;
      ki[j] = PH ? k : KLs[k];
    }
  };
  auto issue_stage = [&](int k0, const int (&ki)[kGC], double (&As)[kTileK][LD], double (&Bs)[kTileK][LD]) {
#pragma unroll
    for (int j = 0; j < kGC; ++j) {
      const int kq = wv * kGC + j;
      const int kk = min(k0 + kq, K2 - 1);
      const int ca = ki[j];
      const int cb = tail ? (ca < nph ? ca + nph : ca - nph) : ca;
      const double *sa = kk < nk ? Am + (long)ca * n : Bm + (long)cb * n;
      const double *sb = kk < nk ? Bm + (long)cb * n : Am + (long)ca * n;
      __builtin_amdgcn_global_load_lds((const IMSRG_G void *)(sa + ra),
                                       (__attribute__((address_space(3))) void *)&As[kq][0], 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const IMSRG_G void *)(sb + rb),
                                       (__attribute__((address_space(3))) void *)&Bs[kq][0], 16, 0, 0);
    }
  };
  // the weight of k' = k0 + t (t < 16) is loaded into a register and only
  // scaled and stored to LDS at the end of the stage
  auto load_w = [&](int k0) -> double {
    const int kk = min(k0 + (int)(threadIdx.x & (kTileK - 1)), K2 - 1);
    const int k = kk < nk ? kk : kk - nk;
    if constexpr (!PH) return kw[k];
    const double w = (double)P.hY * (double)phph[k < nph ? k : k - nph];
    return tail ? w : 1.0;
  };
  auto store_w = [&](int k0, double (&Ws)[kTileK], double w) {
    if (threadIdx.x < kTileK) {
      const int kk = k0 + threadIdx.x;
      Ws[threadIdx.x] = kk >= K2 ? 0.0 : kk < nk ? w : w * h;
    }
  };
  int ki[kGC];
  if (K2 > 0) {  // a channel without pp or hh kets only writes zeros
    load_idx(0, ki);
    issue_stage(0, ki, A0, B0);
    store_w(0, W0, load_w(0));
    load_idx(kTileK, ki);  // clamped: harmless past the end
  }
  __builtin_amdgcn_s_waitcnt(0);  // the copies into LDS have landed
  __syncthreads();
  // one stage: copies of the next stage into (An, Bn, Wn), MFMAs on (Ac, Bc, Wc)
  // mixed precision: FP32 partial sums of the wave's 4 x kGN blocks, flushed into
  // the FP64 accumulators every second stage (32 k)
  flt4 t[4][kGN];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < kGN; ++ni) t[mi][ni] = flt4{0.f, 0.f, 0.f, 0.f};
  auto flush_t = [&]() {
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[mi][ni][q] += (double)t[mi][ni][q];
        t[mi][ni] = flt4{0.f, 0.f, 0.f, 0.f};
      }
  };
  auto stage = [&](int k0, double (&Ac)[kTileK][LD], double (&Bc)[kTileK][LD], double (&Wc)[kTileK],
                   double (&An)[kTileK][LD], double (&Bn)[kTileK][LD], double (&Wn)[kTileK], bool flush) {
    const bool more = k0 + kTileK < K2;
    // loads with register results are unconditional (clamped indices): a
    // branch around them would make the compiler wait for them, and for the
    // copies issued with them, where the paths join
    const double w_next = load_w(k0 + kTileK);
    if (more) issue_stage(k0 + kTileK, ki, An, Bn);
    load_idx(k0 + 2 * kTileK, ki);
    if (!wave_live) {
    } else if constexpr (MIXED) {
#pragma unroll
      for (int ks = 0; ks < kTileK / 4; ++ks) {
        const int kr = ks * 4 + (lane >> 4);
        const double wk = Wc[kr];
        float am[4], bm[kGN], al[4], bl[kGN];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const double a = Ac[kr][wr + m * 16 + (lane & 15)] * wk;
          am[m] = (float)a;
          if constexpr (SPLIT) al[m] = (float)(a - (double)am[m]);
        }
#pragma unroll
        for (int m = 0; m < kGN; ++m) {
          const double b = Bc[kr][wc + m * 16 + (lane & 15)];
          bm[m] = (float)b;
          if constexpr (SPLIT) bl[m] = (float)(b - (double)bm[m]);
        }
#pragma unroll
        for (int mi = 0; mi < 4; ++mi)
#pragma unroll
          for (int ni = 0; ni < kGN; ++ni) {
            if constexpr (SPLIT) {
              t[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(bl[ni], am[mi], t[mi][ni], 0, 0, 0);
              t[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(bm[ni], al[mi], t[mi][ni], 0, 0, 0);
            }
            t[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(bm[ni], am[mi], t[mi][ni], 0, 0, 0);
          }
        // split products flush every 4 k: with the operand rounding gone, the
        // FP32 partial sums over 32 k would set the error
        if constexpr (SPLIT) flush_t();
      }
      if (!SPLIT && flush) flush_t();
    } else {
#pragma unroll
      for (int ks = 0; ks < kTileK / 4; ++ks) {
        const int kr = ks * 4 + (lane >> 4);
        const double wk = Wc[kr];
        // the weight of k scales the kGN B values rather than the four A
        // values (1.8% off the FP64 pp/hh GEMM; the mixed kernel keeps it on A,
        // where moving it costs spills)
        double a[4], b[kGN];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = Ac[kr][wr + m * 16 + (lane & 15)];
#pragma unroll
        for (int m = 0; m < kGN; ++m) b[m] = Bc[kr][wc + m * 16 + (lane & 15)] * wk;
#pragma unroll
        for (int mi = 0; mi < 4; ++mi)
#pragma unroll
          for (int ni = 0; ni < kGN; ++ni)
            acc[mi][ni] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[ni], a[mi], acc[mi][ni], 0, 0, 0);
      }
    }
    if (more) store_w(k0 + kTileK, Wn, w_next);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of the next stage have landed
    __syncthreads();
  };
  for (int k0 = 0; k0 < K2; k0 += 2 * kTileK) {
    stage(k0, A0, B0, W0, A1, B1, W1, false);
    if (k0 + kTileK < K2) stage(k0 + kTileK, A1, B1, W1, A0, B0, W0, true);
  }
  if constexpr (MIXED) flush_t();  // a last stage without its pair
  gemm_epilogue<PH, MIXED>(acc, D, n, R0, S0, alpha, h, B.cc_run, s_ph);
}

// ---------------------------------------------------------------------------
// The same 128x128 SYR2K tiles on bf16 MFMA with three-way split operands
// (mixed precision, "bf16x3").  Each FP64 operand x (A values already scaled
// by their weight w_k) is held as three bf16 values x = p0 + p1 + p2:
// p0 = bf16(fl32(x)), p1 = bf16(fl32(x) - p0) and p2 = bf16(fl32(x - (p0 + p1)))
// from the FP64 residual, so |x - (p0 + p1 + p2)| <= 2^-26 |x| (the FP32
// mixed mode rounds each operand by 2^-24).  A product takes six
// v_mfma_f32_16x16x32_bf16 (p0q0, p0q1, p1q0, p1q1, p0q2, p2q0; the dropped
// p1q2 + p2q1 + p2q2 are <= 2^-26 of it), accumulated in FP32 over one stage
// of 32 k and flushed into the FP64 accumulators after every stage.  bf16
// MFMA runs at 16x the FP32 matrix rate on MI355X, so six products cost
// 3/8 of one FP32 product.
// The ph GEMM's kernel (gemm_tile_b3) splits operands once per tile when a
// stage is staged: each wave loads 8 consecutive k of two rows of one operand
// (16-byte global loads, lanes on consecutive row pairs), splits them in
// registers and stores the three bf16x8 vectors in the MFMA operand layout
// (lane l of a 16-row block reads row l % 16, k octet l / 16: one 16-byte LDS
// read per fragment).  The next stage's global loads are issued before the
// current stage's MFMAs.  The pp/hh GEMM splits its operands once per
// commutator instead (k_pack_pphh, below).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

// LDS of one stage: [operand A/B][piece 0..2][k octet 0..3][row 0..127], 16 bytes each
typedef bf16x8 StageB3[2][3][4][kTileB];

// The FP32 intermediates pass through empty asm statements (no instructions):
// otherwise the compiler fuses the double -> float -> bf16 conversions into one
// correctly rounded double -> bf16 conversion (round-to-odd emulation, eight
// instructions), where any nearby p0 serves, the residuals being exact.
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 b2v __attribute__((ext_vector_type(2)));
// The three pieces of two values (consecutive k of one row) at once: each
// rounding to bf16 is one v_cvt_pk_bf16_f32 for the pair.
__device__ __forceinline__ void split3x2(double x0, double x1, b2v &p0, b2v &p1, b2v &p2) {
  f2v f = {(float)x0, (float)x1};
  asm("" : "+v"(f));
  p0 = __builtin_convertvector(f, b2v);
  const f2v f0 = __builtin_convertvector(p0, f2v);
  p1 = __builtin_convertvector(f - f0, b2v);
  const f2v s01 = f0 + __builtin_convertvector(p1, f2v);  // exact: p0 and p1 span at most 18 bits
  f2v r2 = {(float)(x0 - (double)s01[0]), (float)(x1 - (double)s01[1])};
  asm("" : "+v"(r2));
  p2 = __builtin_convertvector(r2, b2v);
}

__device__ __forceinline__ void gemm_tile_b3(PairArg pa, const int4 *items, int nitems) {
  constexpr int T = kTileB, KS = 32;
  __shared__ __align__(16) StageB3 L0, L1;
  bool tail;
  const int4 it = ph_item(items, nitems, tail);
  if (it.y < 0) return;
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  int n, nk, nph = 0;
  const double *Am, *Bm;
  const signed char *phi = nullptr, *phph = nullptr;
  double alpha, h;
  double *D;
  {
    const int cc = it.y;
    n = B.cc_n[cc];
    nph = B.cc_nph[cc];
    nk = 2 * nph;
    const long xo = B.cc_xoff[cc];
    Am = P.Xt + xo;
    Bm = P.Yt + xo;
    D = P.Zbar + B.cc_zoff[cc] + (tail ? (long)n * n : 0);
    alpha = 1.0;
    h = tail || P.hZ == 1 ? 1.0 : -1.0;
    phi = B.cc_phi + B.cc_kstart[cc];
    phph = B.cc_phph + B.cc_phstart[cc];
  }
  const int R0 = it.z * T, S0 = it.w * T;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __shared__ signed char s_ph[2][T];
  if (threadIdx.x < 2 * T) {
    const int sd = threadIdx.x / T, e = threadIdx.x - sd * T;
    s_ph[sd][e] = tail ? phi[min((sd ? S0 : R0) + e, n - 1)] : 1;
  }
  __syncthreads();  // s_ph
  const int K2 = 2 * nk;
  // loader role of this wave: operand (0: rows R0.. of A-side values, 1: rows
  // S0.. of B-side values), k octet, and the lane's two rows
  const int opnd = wv >> 2, oct = wv & 3;
  const int rbase = opnd ? S0 : R0;
  const int row = min(rbase + 2 * lane, n - 1);  // row, row + 1 (one past a column at most: slack)
  // two register sets: the global loads of a stage are issued two stages
  // before it is computed (one stage of compute between issue and use left the
  // load latency exposed at two waves per SIMD)
  d2u va[8], vb[8];
  // global loads of one stage and the factors of its 8 k slots (the weights on
  // the A side, 1 on the B side, 0 past the end).  Indices and weights are
  // wave-uniform; all their scalar loads are issued before any is used, with
  // no branch between them
  auto load_stage = [&](int k0, d2u (&v)[8], double (&wf)[8]) {
    const int kb = k0 + 8 * oct;
    int kk[8], k[8], ca[8];
    double wr[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      kk[j] = min(kb + j, K2 - 1);
      k[j] = kk[j] < nk ? kk[j] : kk[j] - nk;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      ca[j] = k[j];
      wr[j] = !tail ? 1.0 : (double)P.hY * (double)phph[k[j] < nph ? k[j] : k[j] - nph];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int cb = tail ? (ca[j] < nph ? ca[j] + nph : ca[j] - nph) : ca[j];
      // A side: A(., ca) for kk < nk, else B(., cb); B side the other one
      const bool first = kk[j] < nk;
      const double *src = (first != (opnd != 0)) ? Am + (long)ca[j] * n : Bm + (long)cb * n;
      v[j] = *reinterpret_cast<const d2u *>(src + row);
      const double w = first ? wr[j] : wr[j] * h;
      wf[j] = kb + j >= K2 ? 0.0 : opnd ? 1.0 : w;
    }
  };
  auto store_stage = [&](const d2u (&v)[8], const double (&wf)[8], StageB3 &L) {
    union {
      bf16x8 v8;
      b2v h[4];
    } q[2][3];
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      b2v x0, x1, x2, y0, y1, y2;
      split3x2(v[j].x * wf[j], v[j + 1].x * wf[j + 1], x0, x1, x2);  // row 2 lane
      split3x2(v[j].y * wf[j], v[j + 1].y * wf[j + 1], y0, y1, y2);  // row 2 lane + 1
      q[0][0].h[j / 2] = x0; q[0][1].h[j / 2] = x1; q[0][2].h[j / 2] = x2;
      q[1][0].h[j / 2] = y0; q[1][1].h[j / 2] = y1; q[1][2].h[j / 2] = y2;
    }
    const int r = 2 * lane;
#pragma unroll
    for (int pc = 0; pc < 3; ++pc) {
      L[opnd][pc][oct][r] = q[0][pc].v8;
      L[opnd][pc][oct][r + 1] = q[1][pc].v8;
    }
  };
  const int wr = (wv & 1) * 64, wc = (wv >> 1) * kGW;
  const bool wave_live = tile_wave_live(R0, S0, n, wv);
  dbl4 acc[4][kGN];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < kGN; ++b) acc[a][b] = dbl4{0.0, 0.0, 0.0, 0.0};
  auto compute = [&](const StageB3 &L) {
    if (!wave_live) return;
    const int oc = lane >> 4, rl = lane & 15;
    // the B-side fragments of all three pieces stay in registers; the A side
    // is read one piece at a time (fewer registers live at once)
    bf16x8 bfr[kGN][3];
#pragma unroll
    for (int pc = 0; pc < 3; ++pc)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni) bfr[ni][pc] = L[1][pc][oc][wc + ni * 16 + rl];
    flt4 t[4][kGN];
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni) t[mi][ni] = flt4{0.f, 0.f, 0.f, 0.f};
    // products p_a q_b with a + b <= 2: (2,0), then (1,0), (1,1), then (0,2), (0,1), (0,0);
    // one product for all 8 blocks before the next, so that consecutive MFMAs
    // into one accumulator are 8 instructions apart
#pragma unroll
    for (int pa3 = 2; pa3 >= 0; --pa3) {
      bf16x8 af[4];
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) af[mi] = L[0][pa3][oc][wr + mi * 16 + rl];
#pragma unroll
      for (int pb3 = 2 - pa3; pb3 >= 0; --pb3)
#pragma unroll
        for (int mi = 0; mi < 4; ++mi)
#pragma unroll
          for (int ni = 0; ni < kGN; ++ni)
            t[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[ni][pb3], af[mi], t[mi][ni], 0, 0, 0);
    }
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[mi][ni][q] += (double)t[mi][ni][q];
  };
  if (K2 > 0) {  // a channel without pp or hh kets only writes zeros
    const int nst = (K2 + KS - 1) / KS;
    double wa[8], wb[8];
    load_stage(0, va, wa);
    if (nst > 1) load_stage(KS, vb, wb);
    store_stage(va, wa, L0);
    __syncthreads();
    for (int st = 0; st < nst; st += 2) {
      // stage st in L0, stage st+1 in flight in vb, va free
      if (st + 2 < nst) load_stage((st + 2) * KS, va, wa);
      compute(L0);
      if (st + 1 < nst) store_stage(vb, wb, L1);
      __syncthreads();
      if (st + 1 >= nst) break;
      // stage st+1 in L1, stage st+2 in flight in va, vb free
      if (st + 3 < nst) load_stage((st + 3) * KS, vb, wb);
      compute(L1);
      if (st + 2 < nst) store_stage(va, wa, L0);
      __syncthreads();
    }
  }
  gemm_epilogue<true, true>(acc, D, n, R0, S0, alpha, h, B.cc_run, s_ph);
}

// ---------------------------------------------------------------------------
// Mixed pp/hh GEMM from packed panels.  k_pack_pphh splits each operand element
// once per commutator into its three bf16 pieces (split3x2, X already scaled by
// its weight) and stores them in the MFMA operand layout; the tile kernel then
// fills its LDS stages with direct global->LDS copies of those panels (no
// register staging, no conversion per tile) and runs six bf16 products per
// product as gemm_tile_b3 does.  The SYR2K's two halves are
//   sum_k (X w)(r,k) Y(s,k)  and  h * sum_k Y(r,k) (X w)(s,k),
// so the second half reads the same two panels with the sides swapped and its
// FP32 partial sums are flushed with the factor h.

// one work item: k octet it.z of channel it.y, rows 256 it.w .. + 255
__global__ __launch_bounds__(256) void k_pack_pphh(PairArg pa, const int4 *items) {
  const int4 it = items[blockIdx.x];
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const int ch = it.y, oct = it.z;
  const int n = B.ch_n[ch];
  const int k0s = B.k_start[ch], nk = B.k_start[ch + 1] - k0s;
  const int nrp = (n + kTileB - 1) / kTileB * kTileB;
  const int noct = (nk + kB3K - 1) / kB3K * (kB3K / 8);
  const int r = it.w * 256 + (int)threadIdx.x;
  if (r >= nrp) return;
  const long off = B.ch_off[ch];
  const double *X2 = P.X + B.two_off + off, *Y2 = P.Y + B.two_off + off;
  const int rr = min(r, n - 1);
  double xv[8], yv[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int k = 8 * oct + j;
    const int kc = min(k, nk - 1);
    const int col = B.k_loc[k0s + kc];  // wave-uniform
    const double w = B.k_w[k0s + kc];
    const bool ok = k < nk && r < n;
    const double x = X2[(long)col * n + rr], y = Y2[(long)col * n + rr];
    xv[j] = ok ? x * w : 0.0;
    yv[j] = ok ? y : 0.0;
  }
  union {
    bf16x8 v8;
    b2v h[4];
  } qx[3], qy[3];
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    split3x2(xv[j], xv[j + 1], qx[0].h[j / 2], qx[1].h[j / 2], qx[2].h[j / 2]);
    split3x2(yv[j], yv[j + 1], qy[0].h[j / 2], qy[1].h[j / 2], qy[2].h[j / 2]);
  }
  bf16x8 *px = reinterpret_cast<bf16x8 *>(P.panel) + B.pk_off[ch];
  bf16x8 *py = px + (long)noct * 3 * nrp;
#pragma unroll
  for (int pc = 0; pc < 3; ++pc) {
    px[((long)oct * 3 + pc) * nrp + r] = qx[pc].v8;
    py[((long)oct * 3 + pc) * nrp + r] = qy[pc].v8;
  }
}

// The stream of panels through the L2 into LDS (4.0 GB per commutator at emax = 10) and the
// matrix instructions take about as long as each other: alone, 494 us and 377 us at
// emax = 10, 2.96 and 2.39 ms at emax = 12 (327 us and 1.94 ms for the stream with the tiles
// in super-tile order).  One work-group of two waves per SIMD that waited for its copies,
// read and computed stage by stage took 541 us and 3.49 ms, with the copies two stages ahead
// 541 and 3.38, with the FP64 sums of a stage between the next one's matrix instructions
// 530 and 3.40; with both, the waves in two groups a phase apart and the super-tiles 496 us
// and 3.08 ms (the same phases with two LDS stages: 550 us and 3.55 ms).
// Waits until at most N of this wave's copies into LDS are in flight.
template <int N>
__device__ __forceinline__ void wait_copies() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | N);  // expcnt and lgkmcnt untouched
}
// Work-group barrier that waits for this wave's LDS reads and writes but, unlike
// __syncthreads(), not for its copies from memory into LDS.
__device__ __forceinline__ void barrier_lds() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__global__ __launch_bounds__(kGWaves * 64, 2) void k_pphh_big_b3p(PairArg pa, const int4 *items) {
  constexpr int T = kTileB;
  __shared__ __align__(16) StageB3 L0, L1, L2;  // 3 x 48 KiB: one work-group per CU
  const int4 it = items[blockIdx.x];
  if (it.y < 0) return;  // padding item of the XCD-balanced order
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const int ch = it.y;
  const int n = B.ch_n[ch];
  const int nk = B.k_start[ch + 1] - B.k_start[ch];
  const int nrp = (n + kTileB - 1) / kTileB * kTileB;
  const int noct = (nk + kB3K - 1) / kB3K * (kB3K / 8);
  const bf16x8 *px = reinterpret_cast<const bf16x8 *>(P.panel) + B.pk_off[ch];
  const bf16x8 *py = px + (long)noct * 3 * nrp;
  const double alpha = (double)P.hY, h = (double)P.hZ;
  double *D = P.Z + B.two_off + B.ch_off[ch];
  const int R0 = it.z * T, S0 = it.w * T;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nst1 = noct / 4, nst = 2 * nst1;  // stages of 32 k per half, both halves
  // stage copies: 2 sides x 3 pieces x 4 k octets x 2 halves of 64 rows = 48
  // wave copies of 1 KiB (16 bytes per lane), six per wave
  auto issue = [&](int st, StageB3 &L) {
    const bool second = st >= nst1;
    const int o0 = (second ? st - nst1 : st) * 4;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int q = wv * 6 + i;
      const int side = q / 24, pc = (q / 8) % 3, oct = (q / 2) % 4, half = q & 1;
      const bf16x8 *src = ((side == 0) != second) ? px : py;
      const int row0 = (side ? S0 : R0) + half * 64;
      const bf16x8 *g = src + ((long)(o0 + oct) * 3 + pc) * nrp + row0 + lane;
      __builtin_amdgcn_global_load_lds((const IMSRG_G void *)g,
                                       (__attribute__((address_space(3))) void *)&L[side][pc][oct][half * 64], 16, 0,
                                       0);
    }
  };
  const int wr = (wv & 1) * 64, wc = (wv >> 1) * kGW;
  const bool wave_live = tile_wave_live(R0, S0, n, wv);
  dbl4 acc[4][kGN];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < kGN; ++b) acc[a][b] = dbl4{0.0, 0.0, 0.0, 0.0};
  // A stage in two phases: its operands from LDS into registers, then six bf16 products
  // summed in FP32 (smallest first) into t, while the previous stage's sums u go to the FP64
  // accumulators with their half's factor (1, or h for the second half).  Waves 0..3, one per
  // SIMD, are one phase ahead of waves 4..7: while one wave of a SIMD keeps the matrix unit
  // busy, the other reads.
  bf16x8 bfr[kGN][3], af[3][4];
  auto read = [&](const StageB3 &L) {
    if (!wave_live) return;
    const int oc = lane >> 4, rl = lane & 15;
#pragma unroll
    for (int pc = 2; pc >= 0; --pc) {
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni) bfr[ni][pc] = L[1][pc][oc][wc + ni * 16 + rl];
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) af[pc][mi] = L[0][pc][oc][wr + mi * 16 + rl];
    }
  };
  auto compute = [&](flt4 (&t)[4][kGN], const flt4 (&u)[4][kGN], double fl) {
    if (!wave_live) return;
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni) t[mi][ni] = flt4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int pa3 = 2; pa3 >= 0; --pa3)
#pragma unroll
      for (int pb3 = 2 - pa3; pb3 >= 0; --pb3)
#pragma unroll
        for (int mi = 0; mi < 4; ++mi)
#pragma unroll
          for (int ni = 0; ni < kGN; ++ni)
            t[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[ni][pb3], af[pa3][mi], t[mi][ni], 0, 0, 0);
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[mi][ni][q] += fl * (double)u[mi][ni][q];
    // 48 matrix instructions with the 64 conversions and adds between them
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
  };
  if (nst > 0) {  // a channel without pp or hh kets only writes zeros
    flt4 t0[4][kGN], t1[4][kGN];
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni) t0[mi][ni] = t1[mi][ni] = flt4{0.f, 0.f, 0.f, 0.f};
    auto factor = [&](int st) { return st >= nst1 ? h : 1.0; };
    issue(0, L0);
    issue(1, L1);  // nst is even
    wait_copies<6>();
    barrier_lds();
    if (wv >= 4) barrier_lds();
    // stage st in L.  When it starts, the copies of st have landed in every wave, and every
    // wave has read st - 1, whose buffer Ln takes st + 2; past the end the last stage again,
    // so that six copies are in flight always
    auto stage = [&](int st, const StageB3 &L, StageB3 &Ln, flt4 (&t)[4][kGN], const flt4 (&u)[4][kGN]) {
      issue(min(st + 2, nst - 1), Ln);
      read(L);
      wait_copies<6>();  // those of st + 1
      barrier_lds();
      __builtin_amdgcn_sched_barrier(0);
      compute(t, u, factor(st - 1));
      __builtin_amdgcn_sched_barrier(0);
      barrier_lds();
    };
    for (int st = 0; st < nst; st += 6) {
      stage(st, L0, L2, t0, t1);
      stage(st + 1, L1, L0, t1, t0);
      if (st + 2 >= nst) break;
      stage(st + 2, L2, L1, t0, t1);
      stage(st + 3, L0, L2, t1, t0);
      if (st + 4 >= nst) break;
      stage(st + 4, L1, L0, t0, t1);
      stage(st + 5, L2, L1, t1, t0);
    }
    if (wv < 4) barrier_lds();
    wait_copies<0>();
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[mi][ni][q] += h * (double)t1[mi][ni][q];
  }
  gemm_epilogue<false, true>(acc, D, n, R0, S0, alpha, h, B.cc_run, nullptr);
}

__global__ __launch_bounds__(kGWaves * 64, 2) void k_ph_big_b3(PairArg pa, const int4 *items, int nitems) {
  gemm_tile_b3(pa, items, nitems);
}

__global__ __launch_bounds__(kGWaves * 64, 4) void k_pphh_big_f64(PairArg pa, const int4 *items) {
  gemm_tile<false, false>(pa, items, 0);
}
__global__ __launch_bounds__(kGWaves * 64, 4) void k_pphh_big_mixed(PairArg pa, const int4 *items) {
  gemm_tile<false, true>(pa, items, 0);
}
__global__ __launch_bounds__(kGWaves * 64, 4) void k_pphh_big_split(PairArg pa, const int4 *items) {
  gemm_tile<false, true, true>(pa, items, 0);
}
template <bool SPLIT>
__global__ __launch_bounds__(kGWaves * 64, 4) void k_ph_big(PairArg pa, const int4 *items, int nitems) {
  gemm_tile<true, SPLIT, SPLIT>(pa, items, nitems);
}

// The ph GEMM with FP32 products (gemm_tile's PH = true, MIXED, without SPLIT) on Xbar and
// Ybar^T that the Pandya transformation has stored in FP32.  All its weights are +-1, so that
// rounding the operands there gives the same values as rounding the weighted ones here.
// A stage holds 32 k: with FP64 operands it held 16 in the same LDS, each behind its own
// barrier and with half the time for the copies to arrive.  A 16-byte copy of a wave fills a
// slot of two columns k and k + 4, and slots are 2 x 128 + 16 elements apart: the four k that
// a wave reads at once then lie in different banks and all its reads of a stage are at fixed
// distances from one address.  The FP32 sums are flushed every 32 k.
// emax = 10: 335 -> 254 us, emax = 12: 1461 -> 1145 us (66 -> 85 TF/s on the sub-tiles with
// results), emax = 5: 29 -> 23 us; 26 and 101 us of the first two are the epilogue's.  A tile
// has some 7 stages only, so that its start and its stores take a third of its time.
constexpr int kF32K = 32;
__global__ __launch_bounds__(kGWaves * 64, 4) void k_ph_big_f32(PairArg pa, const int4 *items, int nitems) {
  constexpr int T = kTileB, SL = 2 * T + 16, NS = kF32K / 2;  // slots of two columns
  __shared__ __align__(16) float A0[NS * SL], A1[NS * SL], B0[NS * SL], B1[NS * SL];
  __shared__ signed char s_ph[2][T];
  bool tail;
  const int4 it = ph_item(items, nitems, tail);
  if (it.y < 0) return;  // padding item of the XCD-balanced order
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const int cc = it.y, n = B.cc_n[cc], ld = (n + 3) & ~3, nph = B.cc_nph[cc], nk = 2 * nph, K2 = 2 * nk;
  const IMSRG_G float *Am = (const IMSRG_G float *)(P.Xt + B.cc_xoff[cc]), *Bm = (const IMSRG_G float *)(P.Yt + B.cc_xoff[cc]);
  float *D = reinterpret_cast<float *>(P.Zbar) + B.cc_zoff[cc] + (tail ? (long)n * n : 0);
  const bool hneg = !tail && P.hZ != 1;
  const signed char *phi = B.cc_phi + B.cc_kstart[cc], *phph = B.cc_phph + B.cc_phstart[cc];
  const int R0 = it.z * T, S0 = it.w * T;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x < 2 * T) {
    const int sd = threadIdx.x / T, e = threadIdx.x - sd * T;
    s_ph[sd][e] = tail ? phi[min((sd ? S0 : R0) + e, n - 1)] : 1;
  }
  const int wr = (wv & 1) * 64, wc = (wv >> 1) * kGW;
  const bool wave_live = tile_wave_live(R0, S0, n, wv);
  // copies: lanes 0..31 column k, 32..63 column k + 4 of a slot; four rows per lane, whole
  // quads of a column (its rows n .. ld - 1 and the clamped ones reach no stored result)
  const int ra = min(R0 + 4 * (lane & 31), ld - 4), rb = min(S0 + 4 * (lane & 31), ld - 4);
  auto column = [&](int kk, const IMSRG_G float *&a, const IMSRG_G float *&b) {
    const int ca = kk < nk ? kk : kk - nk, cb = tail ? (ca < nph ? ca + nph : ca - nph) : ca;
    const IMSRG_G float *x = Am + (long)ca * ld, *y = Bm + (long)cb * ld;
    a = kk < nk ? x : y;
    b = kk < nk ? y : x;
  };
  auto issue = [&](int k0, float *As, float *Bs) {
#pragma unroll
    for (int j = 0; j < NS / kGWaves; ++j) {
      const int sl = NS / kGWaves * wv + j, k1 = k0 + 8 * (sl >> 2) + (sl & 3);
      const IMSRG_G float *a1, *b1, *a2, *b2;  // wave-uniform; the lanes choose
      column(min(k1, K2 - 1), a1, b1);
      column(min(k1 + 4, K2 - 1), a2, b2);
      __builtin_amdgcn_global_load_lds((const IMSRG_G void *)((lane < 32 ? a1 : a2) + ra),
                                       (__attribute__((address_space(3))) void *)&As[sl * SL], 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const IMSRG_G void *)((lane < 32 ? b1 : b2) + rb),
                                       (__attribute__((address_space(3))) void *)&Bs[sl * SL], 16, 0, 0);
    }
  };
  // signs of the weights of a stage's k, one bit each: (tail) hY phi of the ph ket, (head) the
  // sign of the second half of the k
  auto load_w = [&](int k0) -> signed char {
    const int kk = min(k0 + (lane & (kF32K - 1)), K2 - 1), k = kk < nk ? kk : kk - nk;
    return phph[k < nph ? k : k - nph];
  };
  auto sign_bits = [&](int k0, signed char w) -> unsigned {
    const bool neg = tail ? (P.hY == 1) != (w > 0) : hneg && k0 + (lane & (kF32K - 1)) >= nk;
    return (unsigned)__ballot(neg);
  };
  dbl4 acc[4][kGN];
  flt4 t[4][kGN];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < kGN; ++b) {
      acc[a][b] = dbl4{0.0, 0.0, 0.0, 0.0};
      t[a][b] = flt4{0.f, 0.f, 0.f, 0.f};
    }
  const int kl = lane >> 4, pa0 = kl * SL + wr + (lane & 15), pb0 = kl * SL + wc + (lane & 15);
  auto step = [&](const float *Ap, const float *Bp, unsigned sg) {
    const unsigned neg = (sg >> kl) << 31;
    float am[4], bm[kGN];
#pragma unroll
    for (int m = 0; m < 4; ++m) am[m] = Ap[16 * m];
#pragma unroll
    for (int m = 0; m < kGN; ++m) bm[m] = __uint_as_float(__float_as_uint(Bp[16 * m]) ^ neg);
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < kGN; ++ni)
        t[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(am[mi], bm[ni], t[mi][ni], 0, 0, 0);
  };
  auto stage = [&](int k0, unsigned sg, const float *As, const float *Bs, float *An, float *Bn) -> unsigned {
    const signed char w_next = load_w(k0 + kF32K);
    if (k0 + kF32K < K2) issue(k0 + kF32K, An, Bn);
    if (wave_live) {
      const int steps = min(kF32K, K2 - k0) >> 2;  // K2 is a multiple of 4
      // not unrolled: more reads ahead than one step's do not fit in the registers
#pragma unroll 1
      for (int ks = 0; ks < steps; ks += 2) {
        const float *Ap = As + pa0 + ks * 2 * SL, *Bp = Bs + pb0 + ks * 2 * SL;
        step(Ap, Bp, sg >> (4 * ks));
        if (ks + 1 < steps) step(Ap + T, Bp + T, sg >> (4 * ks + 4));
      }
#pragma unroll
      for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < kGN; ++ni) {
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[mi][ni][q] += (double)t[mi][ni][q];
          t[mi][ni] = flt4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const unsigned next = sign_bits(k0 + kF32K, w_next);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of the next stage have landed
    __syncthreads();
    return next;
  };
  issue(0, A0, B0);  // K2 > 0: channels with ph kets only
  unsigned sg = sign_bits(0, load_w(0));
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int k0 = 0; k0 < K2; k0 += 2 * kF32K) {
    sg = stage(k0, sg, A0, B0, A1, B1);
    if (k0 + kF32K < K2) sg = stage(k0 + kF32K, sg, A1, B1, A0, B0);
  }
  typedef float f4s __attribute__((ext_vector_type(4), aligned(4)));  // 4-byte aligned columns
  // four consecutive rows of a column per lane: one 16-byte store where all four are stored
  const bool near = S0 + wc - (R0 + wr + 63) < B.cc_run;
  const int run = B.cc_run;
  const double h = hneg ? -1.0 : 1.0;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < kGN; ++ni) {
      const int rr = wr + 16 * mi + 4 * kl, c = wc + 16 * ni + (lane & 15), row = R0 + rr, col = S0 + c;
      if (row >= n || col >= n || row > col) continue;
      const double sc = s_ph[1][c];
      float *dp = D + (long)col * n + row;
      const dbl4 v = acc[mi][ni];
      if (row + 3 < n && row + 3 <= col)
        *reinterpret_cast<f4s *>(dp) = f4s{(float)(sc * v[0]), (float)(sc * v[1]), (float)(sc * v[2]), (float)(sc * v[3])};
      else
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (row + q < n && row + q <= col) dp[q] = (float)(sc * v[q]);
      if (near)  // the lower elements next to the diagonal: h phi_r phi_c times the upper ones
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (row + q < n && row + q < col && col - row - q < run)
            D[(long)(row + q) * n + col] = (float)(h * (double)(s_ph[1][c] * s_ph[0][rr + q]) * (sc * v[q]));
    }
}

// ---------------------------------------------------------------------------
// DoPandyaTransformation_SingleChannel_XandY (src/Commutator.cc:1392-1485):
// Xbar (nk x 2nph) and Ybar^T (nk x 2nph), one element each per thread,
//   Xbar(cd; ab) = -(n_a - n_b) sum_J (2J+1) {ja jb J'; jc jd J} X^J_{cb,ad},
// consecutive threads on consecutive kets cd.  X^J_{cb,ad} is read as hX times the
// element at row (a,d) and column (c,b): for a hole a the rows (a,d) of consecutive d
// are neighbours, where the columns are a whole column apart.  The local indices of
// (c,b) and (a,d) come eight J at a time from 16-byte rows of kmorb, the 6j values two
// J at a time.  Bound by the address processing of its gathers (texture addresser 79%
// busy with one load per index and 6j value and the transposed elements): 182 us at
// emax = 10 before.
__device__ __forceinline__ void front_pandya(const PairPtrs &P, const int4 &it, bool f32, unsigned char *lds_raw) {
  const BasisDev &B = *P.basis;
  // channel offsets and sizes in LDS: the gather of each J then waits on one
  // LDS read instead of two dependent global loads
  int4 *s_ch = (int4 *)lds_raw;
  for (int c = threadIdx.x; c < B.nch; c += blockDim.x) {
    const long off = B.ch_off[c];
    s_ch[c] = make_int4((int)(off & 0xffffffff), (int)(off >> 32), B.ch_n[c], 0);
  }
  __syncthreads();
  const int cc = it.y;
  const int nk = B.cc_n[cc], nph = B.cc_nph[cc];
  const long tot = (long)nk * 2 * nph;
  const long e = (long)it.z + threadIdx.x;
  if (e >= tot) return;
  const int mp = (int)(e / nk), ik = (int)(e % nk);
  const int abc = mp / nph, ibra = mp - abc * nph;
  const int locb = B.cc_ph[B.cc_phstart[cc] + ibra];
  const int kb = B.cc_kets[B.cc_kstart[cc] + locb];
  const int p = B.kp[kb], q = B.kq[kb];
  const int a = abc ? q : p, b = abc ? p : q;
  const int kk = B.cc_kets[B.cc_kstart[cc] + ik];
  const int c = B.kp[kk], d = B.kq[kk];
  const int Jcc = cc / 6;
  const double *X2 = P.X + B.two_off, *Y2 = P.Y + B.two_off;
  double xbar = 0.0, ybar = 0.0, normf = 1.0;
  const double nanb = B.occ[a] - B.occ[b];
  if (B.tz2[a] + B.tz2[d] == B.tz2[b] + B.tz2[c]) {
    if (a == d) normf *= SQRT2_D;
    if (c == b) normf *= SQRT2_D;
    const int ja = B.j2[a], jb = B.j2[b], jc = B.j2[c], jd = B.j2[d];
    const int jmin = max(abs(ja - jd), abs(jc - jb)) / 2;
    const int jmax = min(ja + jd, jc + jb) / 2;
    const int even = a == d || c == b;  // pairs of equal orbits: even J only
    // index work common to X and Y (GetTBME_J_norm_twoOps, src/TwoBodyME.cc:368-409)
    const int pcb = (B.l[c] + B.l[b]) & 1, pad = (B.l[a] + B.l[d]) & 1;
    const int g = 2 * ((B.tz2[c] + B.tz2[b]) / 2 + 1) + pcb;
    if (pcb == pad) {
      const int norb = B.norb, nx = B.kmorb_nx;
      const double *six = B.sixj + sixj_index(B.d1, B.d2, ja, jb, Jcc, jc, jd, 0);
      const IMSRG_G uint4 *k1 = (const IMSRG_G uint4 *)B.kmorb + ((b * norb + c) * nx >> 3);
      const IMSRG_G uint4 *k2 = (const IMSRG_G uint4 *)B.kmorb + ((a * norb + d) * nx >> 3);
      // the swapped kets' phases (-1)^{(j1+j2)/2+1+J}: sign at J = 0 and whether J alternates
      const int s0 = (c > b ? (jc + jb) / 2 + 1 : 0) + (a > d ? (ja + jd) / 2 + 1 : 0);
      const int sj = (c > b) != (a > d);
      for (int c8 = jmin & ~7; c8 <= jmax; c8 += 8) {
        union {
          uint4 v;
          unsigned short s[8];
        } i1, i2;
        i1.v = k1[c8 >> 3];
        i2.v = k2[c8 >> 3];
#pragma unroll
        for (int h = 0; h < 8; h += 4) {
          if (c8 + h > jmax || c8 + h + 3 < jmin) continue;
          typedef double d2s __attribute__((ext_vector_type(2), aligned(8)));
          const d2s w01 = *(const IMSRG_G d2s *)(six + c8 + h), w23 = *(const IMSRG_G d2s *)(six + c8 + h + 2);
          double xv[4], yv[4], wv[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int J = c8 + h + u;
            const unsigned r = i2.s[h + u], cl = i1.s[h + u];  // 0xffff: no such ket
            const double w = u == 0 ? w01.x : u == 1 ? w01.y : u == 2 ? w23.x : w23.y;
            const bool ok = J >= jmin && J <= jmax && !(even & J) && fabs(w) >= 1e-8 && r != 0xffff && cl != 0xffff;
            wv[u] = ok ? (2 * J + 1) * w * sgn_parity(s0 + sj * J) : 0.0;
            // an invalid term is 0 (its address that of the operator's first element)
            const int4 ch = s_ch[ok ? 6 * J + g : 0];
            const long idx = ok ? (((long)ch.y << 32) | (unsigned)ch.x) + (long)(cl * ch.z + r) : 0;
            xv[u] = ok ? X2[idx] : 0.0;
            yv[u] = ok ? Y2[idx] : 0.0;
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            xbar -= wv[u] * xv[u];
            ybar -= wv[u] * yv[u];
          }
        }
      }
      xbar *= P.hX;  // X(cb, ad) = hX X(ad, cb); Ybar^T holds hY Y(cb, ad) = Y(ad, cb)
    }
  }
  if (f32) {  // rounded once, as k_ph_big_f32 would; columns of a multiple of 4 elements
    const long o = (long)mp * ((nk + 3) & ~3) + ik;
    ((IMSRG_G float *)(P.Xt + B.cc_xoff[cc]))[o] = (float)(xbar * normf * nanb);
    ((IMSRG_G float *)(P.Yt + B.cc_xoff[cc]))[o] = (float)(ybar * normf);
    return;
  }
  const long o = B.cc_xoff[cc] + (long)mp * nk + ik;
  P.Xt[o] = xbar * normf * nanb;
  P.Yt[o] = ybar * normf;
}

// First launch of a commutator: the kernels that read only X and Y and write
// scratch, Z1 or Xbar / Ybar, side by side in one grid (work-group ranges in this
// order): zero-body channels, one-body pairs, comm221 partial sums, Pandya chunks.
// Launched one after another they are a chain of four launches of mostly latency
// before the ph GEMM can start (emax = 6: 6 + 18 + 15 + 15 us and the gaps).
__device__ __forceinline__ void front(const PairArg &pa, const FrontItems &f, int b, unsigned char *lds_raw) {
  if (b < f.nzeros) {
    front_zero(pa.get(b / f.nzero), b % f.nzero);
    return;
  }
  b -= f.nzeros;
  if (b < f.none) {
    const int4 it = f.one[b];
    front_one(pa.get(it.x), it);
    return;
  }
  b -= f.none;
  if (b < f.n221) {
    const int4 it = f.ob221[b];
    front_221(pa.get(it.x), it);
    return;
  }
  const int4 it = f.pandya[b - f.n221];
  front_pandya(pa.get(it.x), it, f.xbar_f32, lds_raw);
}
__global__ __launch_bounds__(256, 7) void k_front(PairArg pa, FrontItems f) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  front(pa, f, blockIdx.x, lds_raw);
}

// AddInversePandyaTransformation (src/Commutator.cc:1501-1616), by bra.
//   Z^J_{ij,kl} += f(J) [ sum_J' (2J'+1) {ji jj J; jk jl J'} M^{J'}(l, k)
//                        - (-1)^{(jk+jl)/2 - J} sum_J' (2J'+1) {jj ji J; jk jl J'} M^{J'}(k, l) ] / norm
// with M^{J'}(x, y) = Zbar^{J'}[(ix), (yj)] of the bra (ij); i <= k <= l, so that the rows
// (i, x) of a column follow one another in x.  f(J) stands for the second sum where k = l
// or i = j (1 - (-1)^{(jk+jl)/2 - J}, with (-1)^{(ji+jj+jk+jl)/2} for i = j).
// One work-group per bra, or per range [k0, k1) of its kets' k where the bra's M exceeds
// the LDS of a work-group.  It
//  * lays out M in LDS by sets t = (J', parity and |tz| of (i, x)), each in two blocks: the
//    columns y in [k0, k1) with the rows x >= k0, then the columns y >= k1 with the rows x in
//    [k0, k1); and a table over (J', orbit) of the orbit's column offset and row;
//  * copies M in chunks of 64 elements of one block, each read once;
//  * takes the kets by class (ja <= jb, the unordered j of k and l): the class's weights
//    W(J, J') times the gathered M(J', ket) on the FP64 matrix units, four quads of 4 J x 4
//    kets at once.
//    A ket with jk > jl is its class's with both sums exchanged, which is the factor
//    -(-1)^{(jk+jl)/2 - J} on the result.
// sixjQ holds the weights (2J'+1) {...}, with zeros where the reference skips |6j| < 1e-8.
// CC channels without ph kets (Zbar = 0, not written by the ph GEMM) are read as zeros.
// TZ is the element type of Zbar: float after the FP32-product ph GEMM, double otherwise;
// the sums are FP64.  Every upper element (ij <= kl, or ij < kl for anti-Hermitian Z) of
// every channel is produced exactly once and stored at its transposed slot (row ib of
// channel J, written for this bra only); k_finish adds it to the upper triangle, the
// diagonal is kept apart.
// A lane per ket that gathered its elements from memory (the kernel before this one) read
// the lines again for each class with a ket in them, 3.4 GB at emax = 10 where 0.4 GB are
// needed, and was bound by that: 594 us at emax = 10 FP64, 531 us with FP32 Zbar, 2310 us at
// emax = 12 with FP32 Zbar.  Now 380, 319 and 1303 us; 0.6 GB read.  What bounds it now is
// instruction issue and latency, in about equal parts of the tables, the copies and the
// results: 24 waves per CU, 45% of the cycles with a vector instruction issued.  Tried:
// 16x16x4 matrix instructions on blocks of 16 J x 16 kets (a class of a bra has 13 kets and
// 3.4 J on average): 590 us.
constexpr int kInvpU = 8;    // chunks in flight per wave
constexpr int kInvpW = 2;    // steps of 4 J' whose weights are loaded a block ahead

// inclusive prefix sum over the wave
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// element at a 32-bit byte offset of a (wave-uniform) base
template <class T>
__device__ __forceinline__ T ld_at(const IMSRG_G void *base, unsigned off) {
  return *(const IMSRG_G T *)((const IMSRG_G char *)base + off);
}

template <typename TZ, int kT>
__global__ __launch_bounds__(kT, 6) void k_invpandya(PairArg pa, const int4 *items) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int4 it = items[blockIdx.x];
  if (it.y < 0) return;  // padding item of the XCD-balanced order
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const int i = it.y & 0xFFFF, j = it.y >> 16, k0 = it.z & 0xFFFF, k1 = it.z >> 16, g = it.w >> 28;
  const int nk = B.nkets, norb = B.norb, nJ = B.jmax + 1, nt = B.ccnt, nJp = nt >> 2, ncls = B.ncls;
  const int d1 = B.d1, d2 = B.d2;
  const int norb4 = (norb + 3) & ~3;  // entries of a table row
  const InvpLds L(nJ, nt, norb, ncls, B.invp_nquad, B.invp_nchunk);
  int4 *s_set = (int4 *)(lds_raw + L.set), *s_q = (int4 *)(lds_raw + L.q), *s_z = (int4 *)(lds_raw + L.z);
  int4 *s_cls = (int4 *)(lds_raw + L.cls), *s_sum = s_cls + ncls;
  long *s_row = (long *)(lds_raw + L.row);
  int *s_cf = (int *)(lds_raw + L.cf), *s_pre = (int *)(lds_raw + L.pre);
  unsigned *tabw = (unsigned *)(lds_raw + L.tab);
  const unsigned short *tab = (const unsigned short *)tabw;
  unsigned *s_quad = (unsigned *)(lds_raw + L.quad);
  unsigned short *s_chunk = (unsigned short *)(lds_raw + L.chunk);
  TZ *M = (TZ *)(lds_raw + L.M);
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int nw = kT / 64;
  // the kets elo .. ehi of the group; a range that starts at the bra's own orbit starts at
  // the bra, or after it (anti-Hermitian Z)
  const int elo = (it.w & 0xFFFFFFF) + (k0 == i && P.hZ != 1 ? 1 : 0), ehi = B.grp_first[g * (norb + 1) + k1];
  const int gs = B.grp_start[g];
  const int oi = B.orbcode[i], oj = B.orbcode[j], ji = oi & 0xFFFF, jj = oj & 0xFFFF;
  const bool same = i == j;
  // the table as it is in memory, four orbits per thread: their positions in j's and in i's set
  // at J', or 0xFFFF
  const IMSRG_G uint2 *rkj = (const IMSRG_G uint2 *)(B.cc_rank + (long)j * (nJp + 1) * norb4);
  const IMSRG_G uint2 *rki = (const IMSRG_G uint2 *)(B.cc_rank + (long)i * (nJp + 1) * norb4);
  const int ntab = (nJp + 1) * norb4 >> 2;
  for (int e0 = threadIdx.x; e0 < ntab; e0 += 2 * kT) {
    const int e1 = min(e0 + kT, ntab - 1);
    const uint2 y0 = rkj[e0], x0 = rki[e0], y1 = rkj[e1], x1 = rki[e1];
    uint4 *d = (uint4 *)tabw;
    d[e0] = make_uint4((y0.x & 0xFFFF) | x0.x << 16, y0.x >> 16 | (x0.x & 0xFFFF0000), (y0.y & 0xFFFF) | x0.y << 16,
                       y0.y >> 16 | (x0.y & 0xFFFF0000));
    if (e0 + kT < ntab)
      d[e1] = make_uint4((y1.x & 0xFFFF) | x1.x << 16, y1.x >> 16 | (x1.x & 0xFFFF0000), (y1.y & 0xFFFF) | x1.y << 16,
                         y1.y >> 16 | (x1.y & 0xFFFF0000));
  }
  if (wv == 0) {
    for (int t = lane; t < nt; t += 64) {
      const IMSRG_G unsigned short *ci = B.cc_cnt + (long)i * (norb + 1) * nt + t;
      const IMSRG_G unsigned short *cj = B.cc_cnt + (long)j * (norb + 1) * nt + t;
      const int ci0 = ci[k0 * nt], cj0 = cj[k0 * nt], cii = ci[i * nt];
      int W = ci[norb * nt] - ci0, w = ci[k1 * nt] - ci0;
      const int ns = cj[k1 * nt] - cj0, ny = cj[norb * nt] - cj0;
      if ((t & 2) && !((oi ^ oj) >> 17)) W = w = 0;  // kets of the other Tz
      const int cc = 6 * (t >> 2) + 2 * (((t >> 1) & 1) + 1) + (t & 1), cst = B.cc_cstart[j * nt + t] + cj0;
      const long zo = B.cc_nph[cc] > 0 ? B.cc_zoff[cc] + B.cc_row[i * nt + t] + ci0 - cii : -1;
      s_set[t] = make_int4(ns, cj0, ci0, 0);
      s_q[2 * t] = make_int4(0, W, ns, cst);
      s_q[2 * t + 1] = make_int4(0, w, ny - ns, cst + ns);
      s_z[t] = make_int4((int)(zo & 0xFFFFFFFF), (int)(zo >> 32), B.cc_n[cc], 0);
    }
  } else if (wv == 1) {
    const long kb = ket_index(norb, i, j);
    for (int J = lane; J < nJ + 16; J += 64) {
      const int ib = J < nJ ? B.kmapT[J * (long)nk + kb] : -1;
      s_row[J] = ib < 0 ? -1 : 8 * (B.ch_off[6 * J + g] + (long)ib * B.ch_n[6 * J + g]);
    }
  } else if (wv < 4) {
    for (int c = threadIdx.x - 128; c < ncls; c += 128) {
      const IMSRG_G int *bf = B.cls_before + (long)(gs + g) * ncls + c;
      const int lo = bf[(long)elo * ncls], cnt = elo < ehi ? bf[(long)ehi * ncls] - lo : 0;
      const int jab = B.cls_j[c], ja = jab >> 16, jb = jab & 0xFFFF;
      const int Jlo = max(abs(ji - jj), abs(ja - jb)) / 2, nj = min(ji + jj, ja + jb) / 2 - Jlo + 1;
      const int Dlo = max(abs(ji - jb), abs(jj - ja)) / 2, nD = min(min(ji + jb, jj + ja) / 2, nJp - 1) - Dlo + 1;
      const int Xlo = max(abs(jj - jb), abs(ji - ja)) / 2, nX = min(min(jj + jb, ji + ja) / 2, nJp - 1) - Xlo + 1;
      s_cls[c] = make_int4(B.cls_start[g * ncls + c] + lo, cnt, Jlo | (ja + jb) / 2 << 16, (max(nj, 0) + 3) >> 2);
      // row of the weights at J' = 0 (from that of ja = jb = 1/2), first J' of the two sums, steps of 4 J'
      s_sum[c] = make_int4(((ja >> 1) * d1 + (jb >> 1)) * d2, Dlo, Xlo,
                           (max(max(nD, same ? 0 : nX), 0) + 3) >> 2);
    }
  }
  __syncthreads();
  // prefix sums: element offsets and chunks of the blocks (wave 0), result quads of the classes
  // (wave 1)
  if (wv == 0) {
    int sum = 0;  // chunks << 17 | elements
    for (int q0 = 0; q0 < 2 * nt; q0 += 64) {
      const int q = q0 + lane;
      const int va = q < 2 * nt ? s_q[q].y * s_q[q].z : 0, v = ((va + 63) >> 6) << 17 | va;
      const int p = sum + wave_scan(v);
      if (q < 2 * nt) {
        s_q[q].x = (p - v) & 0x1FFFF;
        s_cf[q] = (p - v) >> 17;
      }
      sum = __builtin_amdgcn_readlane(p, 63);
    }
    if (lane == 0) {
      s_cf[2 * nt] = sum >> 17;
      s_cf[2 * nt + 1] = sum & 0x1FFFF;
    }
  } else if (wv == 1) {
    int sum = 0;
    for (int c0 = 0; c0 < ncls; c0 += 64) {
      const int c = c0 + lane;
      const int v = c < ncls ? ((s_cls[c].y + 3) >> 2) * s_cls[c].w : 0;
      const int p = sum + wave_scan(v);
      if (c < ncls) s_pre[c] = p - v;
      sum = __builtin_amdgcn_readlane(p, 63);
    }
    if (lane == 0) s_pre[ncls] = sum;
  }
  __syncthreads();
  const int nquad = s_pre[ncls], nblk = (nquad + 3) >> 2, nchunk = s_cf[2 * nt];
  const unsigned mz = s_cf[2 * nt + 1];  // the element past M: zero
  if (nblk == 0) return;
  // the table in its final form (each thread its own entries): column offset and row in M,
  // 0xFFFF -- past any element -- where there is none
  for (int e = threadIdx.x; e < ntab; e += kT) {
    const int Jp = (int)(((float)(4 * e) + 2.0f) * __builtin_amdgcn_rcpf((float)norb4)), o4 = 4 * e - Jp * norb4;
    const int4 oc = *(const IMSRG_G int4 *)(B.orbcode + o4);
    uint4 *d = (uint4 *)tabw + e;
    const uint4 v4 = *d;
    auto fin = [&](unsigned v, int oo) -> unsigned {
      const int tx = ((oo ^ oi) >> 16) & 3, ty = ((oo ^ oj) >> 16) & 3;
      const unsigned ry = v & 0xFFFF, rx = v >> 16;
      const int Jc = min(Jp, nJp - 1);
      const int4 st = s_set[4 * Jc + ty];
      const int yr = (int)ry - st.y, part = yr >= st.x;
      const int4 q = s_q[2 * (4 * Jc + ty) + part];
      const unsigned off = ry == 0xFFFF ? ry : (unsigned)(q.x + (yr - (part ? st.x : 0)) * q.y) & 0xFFFF;
      return off | (rx == 0xFFFF ? rx : rx - s_set[4 * Jc + tx].z) << 16;
    };
    if (nJp > 0) *d = make_uint4(fin(v4.x, oc.x), fin(v4.y, oc.y), fin(v4.z, oc.z), fin(v4.w, oc.w));
  }
  for (int q = threadIdx.x; q < 2 * nt; q += kT)
    for (int c = s_cf[q]; c < s_cf[q + 1]; ++c) s_chunk[c] = (unsigned short)q;
  // the result quads: class << 20 | J quad << 15 | ket quad
  for (int c = threadIdx.x; c < ncls; c += kT) {
    const int njq = s_cls[c].w;
    int jq = 0, kq = 0;
    for (int q = s_pre[c]; q < s_pre[c + 1]; ++q) {
      s_quad[q] = c << 20 | jq << 15 | kq;
      if (++jq == njq) {
        jq = 0;
        ++kq;
      }
    }
    if (s_pre[c] < nquad && s_pre[c + 1] == nquad)  // the last block's quads of no ket
      for (int q = nquad; q < 4 * nblk; ++q) s_quad[q] = c << 20 | 0x7FFF;
  }
  if (threadIdx.x == 0) M[mz] = TZ(0);
  __syncthreads();
  // M from Zbar, kInvpU chunks of a wave at once: the columns' indices, then the elements
  for (int c0 = wv; c0 < nchunk; c0 += nw * kInvpU) {
    int col[kInvpU], row[kInvpU], dst[kInvpU], tq[kInvpU];
    TZ z[kInvpU];
#pragma unroll
    for (int u = 0; u < kInvpU; ++u) {
      const int c = min(c0 + u * nw, nchunk - 1);
      const int q = s_chunk[c];
      const int4 a = s_q[q];
      const int m = (c - s_cf[q]) * 64 + lane;
      // m / width: the float quotient is within 1/2 width of the true one (m < 2^16)
      const int yr = (int)(((float)m + 0.5f) * __builtin_amdgcn_rcpf((float)a.y));
      const bool ok = c0 + u * nw < nchunk && yr < a.z;
      row[u] = m - yr * a.y;
      dst[u] = ok ? a.x + m : -1;
      tq[u] = q >> 1;
      col[u] = ld_at<int>(B.cc_cols, 4u * (a.w + (ok ? yr : 0)));
    }
#pragma unroll
    for (int u = 0; u < kInvpU; ++u) {
      const int4 h = s_z[tq[u]];
      const long zo = (((long)h.y << 32) | (unsigned)h.x) + row[u] + (long)((unsigned long)(unsigned)col[u] * (unsigned)h.z);
      const TZ *Zb = reinterpret_cast<const TZ *>(P.Zbar);
      z[u] = Zb[dst[u] >= 0 && h.y >= 0 ? zo : 0];
      if (h.y < 0) z[u] = TZ(0);
    }
#pragma unroll
    for (int u = 0; u < kInvpU; ++u)
      if (dst[u] >= 0) M[dst[u]] = z[u];
  }
  __syncthreads();
  // The results, four quads (4 J x 4 kets of one class) at a time on the 4x4x4 matrix units:
  // lane 16 r + 4 b + m holds row m of the weights of quad b at J' r of a step, the element of
  // its ket m there, and its result of J r and ket m.  The kets' records, their channel indices
  // and the weights of the first kInvpW steps of block bk + nw are loaded before block bk is
  // formed: loaded where they are used they cost most of the time.
  const int rl = lane >> 4, ml = lane & 3;
  struct Blk {
    int Jl, JA, jh;    // the lane's J as a result and as a row of the weights, (ja + jb) / 2
    int pd, px, ns;    // the lane's first J' in the two sums; steps of 4 J'
    int row;           // row of the weights at J' = 0
    bool active;
    int2 rec;
    int ik;
    double wd[kInvpW], wx[kInvpW];
  };
  // held in registers: the stores below could alias B
  const IMSRG_G double *wdir = B.sixjQ + sixjQ_index(d1, d2, ji, jj, 0, 1, 1, 0);
  const IMSRG_G double *wexc = B.sixjQ + sixjQ_index(d1, d2, jj, ji, 0, 1, 1, 0);
  const IMSRG_G int2 *crec = B.cls_rec;
  const IMSRG_G int *ckm = B.cls_kmap;
  IMSRG_G char *Ztwo = (IMSRG_G char *)(P.Z + B.two_off);
  auto weight = [&](const Blk &k, const IMSRG_G double *w, int Jp) -> double {
    return ld_at<double>(w, 8u * ((k.row + min(Jp, nJp)) * d2 + k.JA));
  };
  auto load = [&](int bk) -> Blk {
    Blk k;
    const unsigned q = s_quad[4 * bk + ((lane >> 2) & 3)];
    const int4 k4 = s_cls[q >> 20], c = s_sum[q >> 20];
    const int J0 = (k4.z & 0xFFFF) + (q >> 15 & 31) * 4, p = (q & 0x7FFF) * 4 + ml;
    k.active = p < k4.y;
    const int pos = k4.x + (k.active ? p : 0);
    k.Jl = J0 + rl;
    k.JA = min(J0 + ml, d2 - 1);
    k.jh = k4.z >> 16;
    k.rec = ld_at<int2>(crec, 8u * pos);
    k.ik = ld_at<int>(ckm, 4u * (k.Jl * nk + pos));
    k.row = c.x;
    k.pd = c.y + rl;
    k.px = c.z + rl;
    k.ns = c.w;
#pragma unroll
    for (int u = 0; u < kInvpW; ++u) {  // past the quad's last step: the first one's again
      const int s4 = u < k.ns ? 4 * u : 0;
      k.wd[u] = weight(k, wdir, k.pd + s4);
      k.wx[u] = weight(k, wexc, k.px + s4);
    }
    return k;
  };
  const int brec = ji > jj ? j << 16 | i : i << 16 | j;
  auto form = [&](const Blk &k) {
    const bool sw = k.rec.y != 0;
    const int oa = k.rec.x >> 16, ob = k.rec.x & 0xFFFF;
    const bool dket = oa == ob;
    // first sum: the direct elements M(l, k) of k = oa and l = ob; second: the exchange
    // elements M(k, l), none for k = l.  i = j has the first only, with the true k and l.
    const bool flip = same && sw;
    const int xd = flip ? oa : ob, yd = flip ? ob : oa;
    const unsigned none = dket ? 0xFFFF : 0;
    const double sx = (k.jh - k.JA) & 1 ? 1.0 : -1.0;
    const int ns = max(max(__builtin_amdgcn_readlane(k.ns, 0), __builtin_amdgcn_readlane(k.ns, 4)),
                       max(__builtin_amdgcn_readlane(k.ns, 8), __builtin_amdgcn_readlane(k.ns, 12)));
    double acc = 0.0;
    auto step = [&](int u, double wd, double wx) {
      const int td = min(k.pd + 4 * u, nJp) * norb4, tx = min(k.px + 4 * u, nJp) * norb4;
      const unsigned ed = min((unsigned)tab[2 * (td + yd)] + tab[2 * (td + xd) + 1], mz);
      const unsigned ex = min((unsigned)tab[2 * (tx + ob)] + tab[2 * (tx + oa) + 1] + none, mz);
      const double zd = M[ed], zx = M[ex];
      acc = __builtin_amdgcn_mfma_f64_4x4x4f64(wd, zd, acc, 0, 0, 0);
      if (!same) acc = __builtin_amdgcn_mfma_f64_4x4x4f64(sx * wx, zx, acc, 0, 0, 0);
    };
#pragma unroll
    for (int u = 0; u < kInvpW; ++u)
      if (u < ns) step(u, k.wd[u], k.wx[u]);
    for (int u = kInvpW; u < ns; ++u) step(u, weight(k, wdir, k.pd + 4 * u), weight(k, wexc, k.px + 4 * u));
    const bool odd = (k.jh - k.Jl) & 1;
    double f;
    if (same) {
      const bool oddp = odd != (((ji + jj) / 2 + k.jh) & 1);
      f = dket ? (odd ? 1.0 : 0.0) : oddp ? SQRT2_D : 0.0;
    } else {
      f = dket ? (odd ? SQRT2_D : 0.0) : sw && !odd ? -1.0 : 1.0;
    }
    const long row = s_row[k.Jl];
    if (!k.active || k.ik < 0 || row < 0) return;
    if (k.rec.x == brec)  // diagonal: kept apart (the pp/hh GEMM may still be writing Z's diagonal)
      P.diag[B.ch_kstart[6 * k.Jl + g] + k.ik] = acc * f;
    else
      *(IMSRG_G double *)(Ztwo + (row + 8L * k.ik)) = acc * f;
  };
  // two blocks per turn, so that neither is copied (a copy would wait for its loads)
  Blk ka = load(min(wv, nblk - 1));
  for (int bk = wv; bk < nblk; bk += 2 * nw) {
    const Blk kb2 = load(min(bk + nw, nblk - 1));
    __builtin_amdgcn_sched_barrier(0);
    form(ka);
    if (bk + nw >= nblk) break;
    ka = load(min(bk + 2 * nw, nblk - 1));
    __builtin_amdgcn_sched_barrier(0);
    form(kb2);
  }
}

// The last launch's work-groups before its tile pairs: Z0 (block 0 of a pair) and Z1
// (four one-body pairs each) from the partial sums of the first launch.
__device__ __forceinline__ void finals(const PairArg &pa, int b, int nfin, double *buf, int nbuf) {
  const PairPtrs P = pa.get(b / nfin);
  if (b % nfin == 0) final_zero(P, buf, nbuf);
  else final_one(P, b % nfin - 1);
}

// Lower triangle <- hZ * upper triangle; anti-Hermitian diagonal <- 0.
__global__ __launch_bounds__(256) void k_mirror(PairArg pa, const int4 *items, int nfins, int nfin) {
  __shared__ double t[kTile][kTile + 1];
  if ((int)blockIdx.x < nfins) return finals(pa, blockIdx.x, nfin, &t[0][0], kTile * kTile);
  const int4 it = items[blockIdx.x - nfins];
  if (it.y < 0) return;  // empty item (padding of an XCD run)
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const int ch = it.y, n = B.ch_n[ch];
  const int R0 = it.z * kTile, S0 = it.w * kTile;
  double *Z2 = P.Z + B.two_off + B.ch_off[ch];
  for (int e = threadIdx.x; e < kTile * kTile; e += blockDim.x) {
    const int rr = e & (kTile - 1), cc = e / kTile;
    const int r = R0 + rr, c = S0 + cc;
    if (r < n && c < n) t[cc][rr] = Z2[(long)c * n + r];
  }
  __syncthreads();
  const double hZ = P.hZ;
  for (int e = threadIdx.x; e < kTile * kTile; e += blockDim.x) {
    const int rr = e & (kTile - 1), cc = e / kTile;
    const int row = S0 + rr, col = R0 + cc;
    if (row >= n || col >= n) continue;
    if (row > col)
      Z2[(long)col * n + row] = hZ * t[rr][cc];
    else if (row == col && P.hZ == -1)
      Z2[(long)col * n + row] = 0.0;
  }
}

// Element idx of a channel block through a 32-bit byte offset (global loads and
// stores then take the block base in SGPRs); a block holds < 2^29 doubles.
template <class T>
__device__ __forceinline__ T &blk_at(T *base, unsigned idx) {
  return *(T *)((char *)base + (idx << 3));
}
template <class T>
__device__ __forceinline__ const T &blk_at(const T *base, unsigned idx) {
  return *(const T *)((const char *)base + (idx << 3));
}

// W of comm122ss (src/Commutator.cc:908-926) by column bins:
//   W(r, q) = sum over the partner entries e of ket q of Y2(r, ind_e) x_e - X2(r, ind_e) y_e,
//   x_e = X1(a,o) f, y_e = Y1(a,o) f for the entry's orbits and factor (857-896).
// Every partner of a bin's kets lies in the bin, so W of the bin's columns is the product
//   W = [Y2 X2](rows, bin) [Cx; -Cy]
// with the coefficient matrices Cx, Cy over the bin, built in LDS from the partner
// entries once per work-group (LDS adds; only the ket itself appears twice in a column,
// and a sum of two does not depend on their order).  The
// products run on f64 16x16x4 MFMAs whose A operands come straight from global memory
// (a load takes 16 rows of 4 columns), so X2 and Y2 are read once, with no pass through
// LDS and no barrier between the loads and their use.  Bound by HBM: X2 and Y2 read, W
// written.  Staging the columns in LDS and mixing them there took 258 us at emax = 10 and
// 1412 us at emax = 12 (3.4 and 2.4 TB/s): few work-groups fitted in a CU, each waiting
// for its own staging.  Now 210 and 950 us (4.2 and 3.6 TB/s).
__host__ __device__ inline int c122w_cols(int nc) { return nc <= kC122MaxN ? (nc + 15) & ~15 : 16; }
inline size_t c122w_lds_bytes(int maxbin) {
  const size_t k4 = (size_t)((maxbin + 3) & ~3), full = maxbin <= kC122MaxN ? k4 * c122w_cols(maxbin) : kC122MaxN * kC122MaxN;
  return 16 * std::max(full, 16 * k4) +  // both matrices of a whole bin, or of 16 columns of a larger one
         sizeof(int) * (size_t)maxbin;
}
__device__ __forceinline__ void c122_w_tile(const PairPtrs &P, const int4 &it, unsigned char *lds_raw) {
  constexpr int KF = kC122MaxN / 4;  // A fragments (4 columns each) held at once
  const BasisDev &B = *P.basis;
  const int ch = it.y, n = B.ch_n[ch];
  const int b0 = B.c122_boff[it.z], nc = B.c122_boff[it.z + 1] - b0;
  const int eo = B.c122_beoff[it.z], ne = B.c122_beoff[it.z + 1] - eo;
  const int R0 = (it.w & 0xffff) * kC122Rows;
  // this item's columns: all of the bin's, or 16 of a bin of more than kC122MaxN
  const int ns = c122w_cols(nc), n0 = (it.w >> 16) * 16, nn = min(nc - n0, ns), k4 = (nc + 3) & ~3;
  double *cx = reinterpret_cast<double *>(lds_raw);  // [k4][ns]: coefficients of Y2
  double *cy = cx + k4 * ns;                         // [k4][ns]: of X2
  int *sq = reinterpret_cast<int *>(cy + k4 * ns);  // [nc] the bin's kets
  for (int t = threadIdx.x; t < 2 * k4 * ns; t += blockDim.x) cx[t] = 0.0;
  for (int t = threadIdx.x; t < nc; t += blockDim.x) sq[t] = B.c122_bcols[b0 + t];
  __syncthreads();
  for (int t = threadIdx.x; t < ne; t += blockDim.x) {
    const int4 rec = B.c122_brec[eo + t];
    const int c = (rec.y >> 16) - n0;
    if (c < 0 || c >= nn) continue;
    const double f = __hiloint2double(rec.w, rec.z);
    const int at = (rec.y & 0xffff) * ns + c;
    atomicAdd(&cx[at], P.X[B.one_off + rec.x] * f);
    atomicAdd(&cy[at], -(P.Y[B.one_off + rec.x] * f));
  }
  __syncthreads();
  const long off = B.ch_off[ch];
  const double *X2 = P.X + B.two_off + off, *Y2 = P.Y + B.two_off + off;
  double *W = P.c122w + off;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15, kq = lane >> 4;
  bool bad = false;
  for (int r0 = R0 + 16 * wv; r0 < min(R0 + kC122Rows, n); r0 += 64) {
    const int row = min(r0 + m, n - 1);
    dbl4 acc[kC122MaxN / 16];
#pragma unroll
    for (int j = 0; j < kC122MaxN / 16; ++j) acc[j] = dbl4{0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < k4; k0 += kC122MaxN) {  // once unless the bin is larger
      double ax[KF], ay[KF];
#pragma unroll
      for (int ks = 0; ks < KF; ++ks) {
        if (k0 + 4 * ks >= k4) break;  // uniform
        const unsigned q = (unsigned)sq[min(k0 + 4 * ks + kq, nc - 1)];  // past nc: coefficients 0
        ay[ks] = blk_at(Y2, q * n + row);
        ax[ks] = blk_at(X2, q * n + row);
      }
#pragma unroll
      for (int j = 0; j < kC122MaxN / 16; ++j) {
        if (16 * j >= nn) break;
#pragma unroll
        for (int ks = 0; ks < KF; ++ks) {
          if (k0 + 4 * ks >= k4) break;
          const int c = (k0 + 4 * ks + kq) * ns + 16 * j + m;
          // D^T blocks: lane l, register q holds row (l & 15), column 4 q + (l >> 4)
          acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(cx[c], ay[ks], acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(cy[c], ax[ks], acc[j], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kC122MaxN / 16; ++j) {
      if (16 * j >= nn) break;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = 16 * j + 4 * q + kq;
        if (c < nn && r0 + m < n) blk_at(W, (unsigned)sq[n0 + c] * n + row) = acc[j][q];
      }
    }
    bad = bad || !__builtin_isfinite(acc[0][0]);
  }
  // A row with an Inf or NaN in a column of the bin is not finite in all of its results, the
  // first among them, through products with 0: the wave's rows with such a result again from
  // their partner entries alone, each lane the columns that it has stored.
  if (!__any(bad)) return;
  for (int row = R0 + 16 * wv + m; row < min(R0 + kC122Rows, n); row += 64) {
    if (__builtin_isfinite(blk_at(W, (unsigned)sq[n0 + min(kq, nn - 1)] * n + row))) continue;
    for (int c = kq; c < nn; c += 4) blk_at(W, (unsigned)sq[n0 + c] * n + row) = 0.0;
    double w = 0.0;
    int last = -1;  // entries of one column follow one another
    for (int t = 0; t < ne; ++t) {
      const int4 rec = B.c122_brec[eo + t];
      const int c = (rec.y >> 16) - n0;
      if (c < 0 || c >= nn || (c & 3) != kq) continue;
      if (c != last) w = 0.0;
      last = c;
      const double f = __hiloint2double(rec.w, rec.z);
      const unsigned e = (unsigned)sq[rec.y & 0xffff] * n + row;
      w += blk_at(Y2, e) * (P.X[B.one_off + rec.x] * f) - blk_at(X2, e) * (P.Y[B.one_off + rec.x] * f);
      blk_at(W, (unsigned)sq[n0 + c] * n + row) = w;
    }
  }
}
__global__ __launch_bounds__(256, 4) void k_c122_w(PairArg pa, const int4 *items) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int4 it = items[blockIdx.x];
  c122_w_tile(pa.get(it.x), it, lds_raw);
}

// The first launch of small bases: their comm122 W items and 64x64 pp/hh tiles, which wait
// for nothing either, beside the others.
template <bool MIXED>
__global__ __launch_bounds__(256, 4) void k_front_small(PairArg pa, FrontItems f) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  int b = blockIdx.x;
  if (b < f.n64) return syr2k_tile<0, MIXED>(pa, f.pphh64[b]);
  b -= f.n64;
  if (b < f.nc122) {
    const int4 it = f.c122[b];
    return c122_w_tile(pa.get(it.x), it, lds_raw);
  }
  front(pa, f, b - f.nc122, lds_raw);
}

// 16-byte access to elements idx, idx + 1 of a channel block (8-byte aligned)
__device__ __forceinline__ double2 blk_ld2(const double *base, unsigned idx) {
  return *reinterpret_cast<const double2 *>(&blk_at(base, idx));
}
__device__ __forceinline__ void blk_st2(double *base, unsigned idx, double2 v) {
  *reinterpret_cast<double2 *>(&blk_at(base, idx)) = v;
}

// Last kernel of a commutator, over the tile pairs of every two-body block:
//   FOLD: upper triangle += the transposed-slot contributions of k_invpandya,
//         diagonal += its diagonal terms (kept in P.diag);
//   C122: comm122ss (src/Commutator.cc:837-932), Z2 -= W + hZ W^T, with W
//         formed beforehand by k_c122_w;
// then lower triangle <- hZ * upper triangle; anti-Hermitian diagonal <- 0.
// Tile pair: U = rows R0.., cols S0.. (R0 <= S0) and its transposed position.
// U stays in registers, two rows per thread in 8 of the wave's 16 columns.  The
// contributions held at the transposed position go through LDS, two rows per
// thread of 8 of the wave's 16 columns R0 + rr of Z2.  Loads and stores of
// Z2 then move 16 bytes per lane (address processing per instruction, not
// bytes, bounds these accesses).
template <bool FOLD, bool C122>
__global__ __launch_bounds__(256, 4) void k_finish(PairArg pa, const int4 *items, int nfins, int nfin) {
  __shared__ double t[kTile][kTile + 1];  // t[rr][cc]: contribution to upper (R0 + rr, S0 + cc)
  if ((int)blockIdx.x < nfins) return finals(pa, blockIdx.x, nfin, &t[0][0], kTile * kTile);
  const int4 it = items[blockIdx.x - nfins];
  if (it.y < 0) return;  // empty item (padding of an XCD run)
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const int ch = it.y, n = B.ch_n[ch];
  const int R0 = it.z * kTile, S0 = it.w * kTile;
  const long off = B.ch_off[ch];
  double *Z2 = P.Z + B.two_off + off;
  const double *W2 = P.c122w + off;                    // comm122 W of this channel (k_c122_w)
  const IMSRG_G double *dg = P.diag + B.ch_kstart[ch];  // inverse-Pandya diagonal terms of this channel
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // lane (h, p): rows p2, p2 + 1 (p2 = 2p) of the tile, in the columns (U) or
  // rows (T) wv + 4 (2 j + h), j < kPairs: two elements per load and store
  const int h = lane >> 5, p2 = 2 * (lane & 31);
  const double hZ = P.hZ;
  constexpr int kPairs = kTile * kTile / 512;
  double2 u[kPairs];
#pragma unroll
  for (int j = 0; j < kPairs; ++j) {  // upper elements (R0 + p2 (+1), S0 + cc)
    const int cc = wv + 4 * (2 * j + h), r = R0 + p2, c = S0 + cc;
    // clamped: no branch around the load (a pair may read one element past its column)
    const double2 z = blk_ld2(Z2, (unsigned)(min(c, n - 1) * n + min(r, n - 1)));
    u[j].x = (r < n && c < n) ? z.x : 0.0;
    u[j].y = (r + 1 < n && c < n) ? z.y : 0.0;
    if (C122) {  // Z2 -= W at the upper element
      const double2 w = blk_ld2(W2, (unsigned)(min(c, n - 1) * n + min(r, n - 1)));
      u[j].x -= w.x;
      u[j].y -= w.y;
    }
  }
#pragma unroll
  for (int j = 0; j < kPairs; ++j) {  // transposed positions (S0 + p2 (+1), R0 + rr)
    const int rr = wv + 4 * (2 * j + h), r = R0 + rr, c = S0 + p2;
    double2 v = {0.0, 0.0};
    if (FOLD) {
      const double2 z = blk_ld2(Z2, (unsigned)(min(r, n - 1) * n + min(c, n - 1)));
      v.x = (r < n && c < n && c != r) ? z.x : 0.0;
      v.y = (r < n && c + 1 < n && c + 1 != r) ? z.y : 0.0;
    }
    if (C122) {  // and -= hZ W at the transposed position
      const double2 w = blk_ld2(W2, (unsigned)(min(r, n - 1) * n + min(c, n - 1)));
      v.x -= hZ * w.x;
      v.y -= hZ * w.y;
    }
    t[rr][p2] = v.x;
    t[rr][p2 + 1] = v.y;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPairs; ++j) {
    const int cc = wv + 4 * (2 * j + h), r = R0 + p2, c = S0 + cc;
    double2 v = {u[j].x + t[p2][cc], u[j].y + t[p2 + 1][cc]};
    const bool ok0 = r < n && c < n && r <= c, ok1 = r + 1 < n && c < n && r + 1 <= c;  // ok1 implies ok0
    // diagonal elements inside the block only: dg holds n entries of this channel
    if (ok0 && r == c) v.x = (P.hZ == -1) ? 0.0 : v.x + (FOLD ? dg[r] : 0.0);
    if (ok1 && r + 1 == c) v.y = (P.hZ == -1) ? 0.0 : v.y + (FOLD ? dg[r + 1] : 0.0);
    if (ok1)
      st_nt2(&blk_at(Z2, (unsigned)(c * n + r)), v.x, v.y);
    else if (ok0)
      st_nt(&blk_at(Z2, (unsigned)(c * n + r)), v.x);
    u[j] = v;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPairs; ++j) {  // new upper values to the threads writing their mirror
    const int cc = wv + 4 * (2 * j + h);
    t[p2][cc] = u[j].x;
    t[p2 + 1][cc] = u[j].y;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPairs; ++j) {  // lower elements (S0 + p2 (+1), R0 + rr) = hZ * upper
    const int rr = wv + 4 * (2 * j + h), r = R0 + rr, c = S0 + p2;
    const bool ok0 = r < n && c < n && r < c, ok1 = r < n && c + 1 < n && r < c + 1;
    const double2 v = {hZ * t[rr][p2], hZ * t[rr][p2 + 1]};
    if (ok0 && ok1)
      st_nt2(&blk_at(Z2, (unsigned)(r * n + c)), v.x, v.y);
    else if (ok0)
      st_nt(&blk_at(Z2, (unsigned)(r * n + c)), v.x);
    else if (ok1)
      st_nt(&blk_at(Z2, (unsigned)(r * n + c + 1)), v.y);
  }
}

// Z2 <- 0 over whole tiles (used when the pp/hh term is switched off)
__global__ __launch_bounds__(256) void k_zero_two(PairArg pa, const int4 *items) {
  const int4 it = items[blockIdx.x];
  if (it.y < 0) return;  // empty item (padding of an XCD run)
  PairPtrs P = pa.get(it.x);
  const BasisDev &B = *P.basis;
  const int ch = it.y, n = B.ch_n[ch];
  const int R0 = it.z * kTile, S0 = it.w * kTile;
  double *Z2 = P.Z + B.two_off + B.ch_off[ch];
  for (int e = threadIdx.x; e < kTile * kTile; e += blockDim.x) {
    const int r = R0 + (e & (kTile - 1)), c = S0 + e / kTile;
    if (r < n && c < n) {
      Z2[(long)c * n + r] = 0.0;
      Z2[(long)r * n + c] = 0.0;
    }
  }
}

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_set_pairs(PairPtrs *tab, PairOps ops) {
  const int i = threadIdx.x;
  if (i >= ops.n) return;
  PairPtrs &p = tab[i];
  p.X = (const IMSRG_G double *)ops.op[i].X;
  p.Y = (const IMSRG_G double *)ops.op[i].Y;
  p.Z = (IMSRG_G double *)ops.op[i].Z;
  p.hX = ops.op[i].hX;
  p.hY = ops.op[i].hY;
  p.hZ = ops.op[i].hZ;
  p.mask = ops.op[i].mask;
}
hipError_t launch_set_pairs(PairPtrs *tab, const PairOps &ops, hipStream_t s) {
  static_assert(PairOps::kMax <= 64, "one thread per pair");
  hipLaunchKernelGGL(k_set_pairs, dim3(1), dim3(64), 0, s, tab, ops);
  return hipGetLastError();
}

hipError_t launch_front(const PairArg &pa, const FrontItems &f, int maxnch, int maxbin, bool mixed64, hipStream_t s) {
  size_t lds = sizeof(int4) * (size_t)std::max(maxnch, 1);  // the Pandya chunks' channel table
  if (f.n64 + f.nc122 > 0) {
    if (f.nc122 > 0) lds = std::max(lds, c122w_lds_bytes(maxbin));
    const dim3 grid(f.blocks());
    if (mixed64)
      hipLaunchKernelGGL(k_front_small<true>, grid, dim3(256), lds, s, pa, f);
    else
      hipLaunchKernelGGL(k_front_small<false>, grid, dim3(256), lds, s, pa, f);
    return hipGetLastError();
  }
  FrontItems part[2] = {f, f};
  if (f.split) {
    part[0].npandya = 0;
    part[1].nzeros = part[1].none = part[1].n221 = 0;
  } else {
    part[1].nzeros = part[1].none = part[1].n221 = part[1].npandya = 0;
  }
  for (const FrontItems &p : part)
    if (p.blocks() > 0) hipLaunchKernelGGL(k_front, dim3(p.blocks()), dim3(256), lds, s, pa, p);
  return hipGetLastError();
}
hipError_t launch_pphh(const PairArg &pa, const int4 *items, int nitems, const int4 *items64, int nitems64,
                       const int4 *pack, int npack, int precision, int maxn, hipStream_t s) {
  if (nitems > 0) {
    const size_t lds = sizeof(int) * (size_t)std::max(maxn, 1);  // column-index list of the largest channel
    if (precision == kGemmB3) {
      if (npack > 0) hipLaunchKernelGGL(k_pack_pphh, dim3(npack), dim3(256), 0, s, pa, pack);
      hipLaunchKernelGGL(k_pphh_big_b3p, dim3(nitems), dim3(kGWaves * 64), 0, s, pa, items);
    }
    else if (precision == 1)
      hipLaunchKernelGGL(k_pphh_big_mixed, dim3(nitems), dim3(kGWaves * 64), lds, s, pa, items);
    else if (precision == 2)
      hipLaunchKernelGGL(k_pphh_big_split, dim3(nitems), dim3(kGWaves * 64), lds, s, pa, items);
    else
      hipLaunchKernelGGL(k_pphh_big_f64, dim3(nitems), dim3(kGWaves * 64), lds, s, pa, items);
  }
  if (nitems64 > 0) {  // split and bf16x3 products take FP64 64x64 tiles
    if (precision == 1)
      hipLaunchKernelGGL((k_syr2k<0, true>), dim3(nitems64), dim3(256), 0, s, pa, items64);
    else
      hipLaunchKernelGGL((k_syr2k<0, false>), dim3(nitems64), dim3(256), 0, s, pa, items64);
  }
  return hipGetLastError();
}
hipError_t launch_ph_gemm(const PairArg &pa, const int4 *items, int nitems, int precision, bool big, hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (big) {
    const dim3 grid((nitems + 7) / 8 * 16), blk(kGWaves * 64);  // head and tail of every item (ph_item)
    if (precision == kGemmB3)
      hipLaunchKernelGGL(k_ph_big_b3, grid, blk, 0, s, pa, items, nitems);
    else if (precision == 1)
      hipLaunchKernelGGL(k_ph_big_f32, grid, blk, 0, s, pa, items, nitems);
    else if (precision == 2)
      hipLaunchKernelGGL((k_ph_big<true>), grid, blk, 0, s, pa, items, nitems);
    else
      hipLaunchKernelGGL((k_ph_big<false>), grid, blk, 0, s, pa, items, nitems);
    return hipGetLastError();
  }
  if (precision == 1) {
    hipLaunchKernelGGL((k_syr2k<1, true>), dim3(nitems), dim3(256), 0, s, pa, items);
    hipLaunchKernelGGL((k_syr2k<2, true>), dim3(nitems), dim3(256), 0, s, pa, items);
  } else {
    hipLaunchKernelGGL((k_syr2k<1, false>), dim3(nitems), dim3(256), 0, s, pa, items);
    hipLaunchKernelGGL((k_syr2k<2, false>), dim3(nitems), dim3(256), 0, s, pa, items);
  }
  return hipGetLastError();
}
hipError_t launch_invpandya(const PairArg &pa, const int4 *items, int nitems, size_t lds, bool zbar_f32,
                            hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  // 256 threads where five and more work-groups fit in a CU: 512 take longer on small items
  // (emax = 5, FP32 Zbar: 23.7 against 19.2 us, 48 pairs at emax 4-7 998 against 635 us) and less
  // on large ones (emax = 10, FP64: 383 against 452 us), of which few fit
  const bool small = lds <= kInvpLdsSmall[1];
  const dim3 grid(nitems), blk(small ? 256 : 512);
  if (zbar_f32 && small)
    hipLaunchKernelGGL((k_invpandya<float, 256>), grid, blk, lds, s, pa, items);
  else if (zbar_f32)
    hipLaunchKernelGGL((k_invpandya<float, 512>), grid, blk, lds, s, pa, items);
  else if (small)
    hipLaunchKernelGGL((k_invpandya<double, 256>), grid, blk, lds, s, pa, items);
  else
    hipLaunchKernelGGL((k_invpandya<double, 512>), grid, blk, lds, s, pa, items);
  return hipGetLastError();
}
hipError_t launch_finish(const PairArg &pa, const int4 *items, int nitems, bool fold, bool c122, int npairs,
                         int maxn1pairs, hipStream_t s) {
  const int nfin = 1 + (maxn1pairs + 3) / 4;  // work-groups of final_zero and final_one per pair
  const int nfins = npairs * nfin;
  const dim3 grid(nfins + nitems);
  if (fold && c122)
    hipLaunchKernelGGL((k_finish<true, true>), grid, dim3(256), 0, s, pa, items, nfins, nfin);
  else if (fold)
    hipLaunchKernelGGL((k_finish<true, false>), grid, dim3(256), 0, s, pa, items, nfins, nfin);
  else if (c122)
    hipLaunchKernelGGL((k_finish<false, true>), grid, dim3(256), 0, s, pa, items, nfins, nfin);
  else
    hipLaunchKernelGGL(k_mirror, grid, dim3(256), 0, s, pa, items, nfins, nfin);
  return hipGetLastError();
}
hipError_t launch_c122_w(const PairArg &pa, const int4 *items, int nitems, int maxbin, hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  const size_t lds = c122w_lds_bytes(maxbin);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_c122_w, dim3(nitems), dim3(256), lds, s, pa, items);
  return hipGetLastError();
}
hipError_t launch_zero_two(const PairArg &pa, const int4 *items, int nitems, hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_two, dim3(nitems), dim3(256), 0, s, pa, items);
  return hipGetLastError();
}

}  // namespace imsrg
