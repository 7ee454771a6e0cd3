// internal.hpp -- device-side tables, operator addressing and work items shared
// by the host driver (api.cpp, basis.cpp) and the HIP kernels (*.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace imsrg {

// Pointer members of the structs below address global memory.  In the device
// pass they carry address space 1, so that every load and store through them
// (and through pointers derived from them) compiles to global_* instructions:
// flat_* ones would also count against the LDS wait counter and serialize LDS
// reads with outstanding global loads.  Host code fills the same layout.
#if defined(__HIP_DEVICE_COMPILE__)
#define IMSRG_G __attribute__((address_space(1)))
#else
#define IMSRG_G
#endif

constexpr int kTile = 64;         // SYR2K output tile edge
constexpr int kTileB = 128;       // output tile edge of the large pp/hh SYR2K
constexpr int kTileK = 16;        // k-depth of one LDS stage
constexpr int kGWaves = 8;        // waves of a 128x128 GEMM work-group (2 x 4 grid of 64 x kGW sub-tiles)
constexpr int kGW = 32;           // columns of a wave's sub-tile in the 128x128 GEMM
constexpr int kGN = kGW / 16;     // 16-column MFMA blocks per wave sub-tile
constexpr int kGC = kTileK / kGWaves;  // k columns each wave copies into LDS per stage
constexpr int kChunk = 256;       // elements per work item of the gather kernels
constexpr int kLdsUnit = 1280;    // LDS allocation unit in bytes, 128 of them in a CU
constexpr int kInvpLds = 42 * kLdsUnit;  // LDS of an inverse Pandya work-group: three in a CU
// ... or of one of a small basis, six or five in a CU, with 256 threads instead of 512 (the
// serial parts of more items run at once): FP64 emax = 6 33 -> 29 us, emax = 7 55 -> 46, emax = 8
// 97 -> 92, FP32 Zbar emax = 7 53 -> 45, emax = 8 93 -> 83, emax = 9 171 -> 161.  Where many more bras
// have to be taken in parts it is slower: FP64 emax = 9 184 -> 197, FP32 emax = 10 320 -> 338.
constexpr int kInvpLdsSmall[] = {21 * kLdsUnit, 25 * kLdsUnit};
constexpr int kC122MaxN = 64;     // columns of a comm122 bin formed at once (a larger bin takes one item per 16)
constexpr int kC122MaxCols = 150; // largest bin (LDS: 1 KiB of coefficients per ket)
constexpr int kC122Rows = 128;    // rows of one comm122 W item (256: 221 against 210 us at emax = 10)
constexpr int kXfRows = 128;      // rows of one item of the basis transformation's passes
constexpr int kXfMaxM = 80;       // kets of its largest group (their fragments are held in registers)
constexpr int kF32Flush = 4;      // MFMA k-steps (of 4) summed in FP32 before the FP64 flush (mixed, 64x64 tiles)

// GEMM kernel families passed to launch_pphh / launch_ph_gemm: 0 FP64,
// 1 FP32 MFMA on FP32-rounded operands, 2 split FP32 products, kGemmB3 bf16
// MFMA on three-way split operands
constexpr int kGemmB3 = 3;
constexpr int kB3K = 32;          // k-depth of one stage of the bf16x3 GEMMs (one v_mfma_f32_16x16x32_bf16)

// Term bits (same values as IMSRG_COMM* in include/imsrg_hip.h)
constexpr unsigned M110 = 1u << 0, M220 = 1u << 1, M111 = 1u << 2, M121 = 1u << 3, M221 = 1u << 4,
                   M122 = 1u << 5, MPPHH = 1u << 6, MPH = 1u << 7;

// All basis tables of one model space, device pointers.  Index conventions:
//  * global ket k of orbits p<=q: k = p(2 norb - 1 - p)/2 + q   (ModelSpace::Index2)
//  * standard channel ch = 6J + 2(Tz+1) + parity, J = 0..jmax  (GetTwoBodyChannelIndex)
//  * cross-coupled channel uses the same formula with Tz = |tz_p - tz_q|/2
//  * kmap[k*(jmax+1)+J]: local index of ket k in the standard channel of
//    angular momentum J with the ket's parity and Tz, or -1
struct BasisDev {
  int norb, nkets, nch, jmax, d1, d2;
  int nholes, n1pairs;
  long tbsize;   // doubles in the two-body arena
  long one_off;  // offset of the one-body block inside an operator buffer
  long two_off;  // offset of the two-body arena inside an operator buffer
  long opsize;   // doubles per operator buffer (including 8 doubles of zero slack at the end)
  int maxn, maxblk;
  int ccjmax_ph;  // largest J of a CC channel with ph kets (-1: none); Zbar is zero above it
  const IMSRG_G int *j2, *l, *tz2, *cvq;
  const IMSRG_G int *orbcode;   // j2 | (l & 1) << 16 | (tz2 > 0) << 17, norb4 = norb rounded up to 4 entries
  const IMSRG_G double *occ;
  const IMSRG_G int *holes;
  const IMSRG_G int *obstart, *oblist;  // one-body block of each orbit
  const IMSRG_G int *kp, *kq;
  const IMSRG_G int *kmap;
  const IMSRG_G int *kmapT;     // kmapT[J*nkets + k] = kmap[k*(jmax+1) + J]
  // the cross-coupled kets of one orbit o, by t = 4J + 2|tz_o - tz_x|/2 + parity for J <= ccjmax_ph
  // (ccnt = 4 (ccjmax_ph + 1) such sets), in the order of the other orbit x:
  const IMSRG_G unsigned short *cc_cnt;   // cc_cnt[(o*(norb+1) + k)*ccnt + t]: orbits x < k of set t
  const IMSRG_G unsigned short *cc_rank;  // cc_rank[(o*(ccjmax_ph+2) + J)*norb4 + x]: position of x, or 0xFFFF
  const IMSRG_G int *cc_row;    // cc_row[o*ccnt + t]: local index of the first ket (o, x >= o), the others follow
  const IMSRG_G int *cc_cstart; // cc_cols[cc_cstart[o*ccnt + t] ..]: columns of Zbar, the local index of
  const IMSRG_G int *cc_cols;   //   ket (x, o), plus the channel's size (its tail) for x > o
  int ccnt, cc_run;             // cc_run: most kets of one channel with the same first orbit
  // kmorb[(x*norb + y)*kmorb_nx + J]: standard local index of the ket of orbits x and y at J, 0xffff
  // for none; kmorb_nx: jmax + 1 rounded up to a multiple of 8
  const IMSRG_G unsigned short *kmorb;
  int kmorb_nx;
  // kets of each (parity, Tz) group g = 2(Tz+1) + parity (the channels 6J + g), in ascending
  // global index one group after another: group g's start at position grp_start[g]
  const IMSRG_G int *grp_start;
  const IMSRG_G int *grp_first;  // grp_first[g*(norb+1) + k]: first ket of group g with an orbit p >= k
  // standard channels
  const IMSRG_G long *ch_off;
  const IMSRG_G int *ch_n, *ch_kstart, *ch_kets;
  const IMSRG_G double *w220;  // per channel ket: (1-n_p)(1-n_q) for hh/ph kets, 1 for pp kets
  const IMSRG_G int *hh_start, *hh_loc;
  const IMSRG_G double *hh_occ;
  const IMSRG_G int *k_start, *k_loc;  // pp/hh product list with combined weight (w_pp - w_hh)
  const IMSRG_G double *k_w;
  // bf16x3 operand panels of the mixed pp/hh GEMM (16-byte units): channel ch
  // starts at pk_off[ch] with the panel of X W, then the panel of Y, each
  // [nkp/8 k octets][3 pieces][nrp rows] (nkp = nk rounded up to kB3K, nrp = n
  // rounded up to kTileB); pk_size units in all
  const IMSRG_G long *pk_off;
  long pk_size;
  const IMSRG_G int *kpp_start, *kpp_loc;  // M_pp list (weights w_pp)
  const IMSRG_G double *kpp_w;
  const IMSRG_G int *khh_start, *khh_loc;  // M_hh list (weights n_p n_q)
  const IMSRG_G double *khh_w;
  // comm122 column bins (kets of whole one-body block pairs, closed under
  // partners): bin b holds the channel-local kets c122_bcols[c122_boff[b] ..
  // c122_boff[b + 1]).  The partner entries of its columns, one after another, are the
  // records c122_brec[c122_beoff[b] ..] = (index a + o norb of the one-body element,
  // column << 16 | position of the partner, both in the bin, the factor f -- phase /
  // sqrt2 factors, times 2 for kets with p == q -- as low and high word)
  const IMSRG_G int *c122_bcols;
  const IMSRG_G int *c122_boff;
  const IMSRG_G int4 *c122_brec;
  const IMSRG_G int *c122_beoff;
  int c122_maxbin;                 // kets of the largest bin
  // cross-coupled channels
  const IMSRG_G int *cc_n, *cc_nph, *cc_kstart, *cc_kets, *cc_phstart, *cc_ph;
  const IMSRG_G signed char *cc_phi;  // (-1)^{(j_p+j_q)} per CC ket
  const IMSRG_G signed char *cc_phph; // cc_phi of the ket at each position of the cc_ph lists
  const IMSRG_G long *cc_xoff, *cc_zoff;
  long xsize, zsize;
  // kets of each (parity, Tz) group g by the class c of their unordered pair of j, ja <= jb
  // (cls_j[c] = ja << 16 | jb, as 2j): positions cls_start[g ncls + c] .. of the lists below,
  // ascending kets; cls_before[(grp_start[g] + g + e) ncls + c]: those among the first e kets
  const IMSRG_G int *cls_j, *cls_start, *cls_before;
  const IMSRG_G int2 *cls_rec;  // (a << 16 | b, 1 if the ket is (b, a)): its orbits of ja and jb
  const IMSRG_G int *cls_kmap;  // cls_kmap[J nkets + position]: local index at J or -1, J <= jmax + 16
  int ncls;
  int invp_nquad, invp_nchunk;  // most result quads and 64-element chunks of an inverse Pandya item
  const IMSRG_G int2 *pairs1;   // one-body pairs (i<=j, same (l,j2,tz2) block)
  // partial sums of the one-body part: slots ob_start[p] .. ob_start[p+1]-1 of pair p
  // (the first: comm111 + comm121, the others: comm221 items); cpart: orbits with 1 - n_c != 0;
  // ob_cj: c << 8 | J of each pair's orbits c with n_c != 0
  const IMSRG_G int *ob_start, *cpart, *ob_cj;
  int nobpart, ncpart;
  int ndiag;  // kets summed over all channels (ch_kstart[nch])
  const IMSRG_G double *w1norm; // norb*norb one-body norm weights
  const IMSRG_G double *sixj;   // dense 6j table, layout of SixJCache_112112
  const IMSRG_G double *sixjQ;  // (2 J6 + 1) times the values (0 where |6j| < 1e-8), layout
                                // [jj1][jj2][jj4][jj5][J6][J3] (sixjQ_index)
  // generator lists: per channel, core-core kets and (non-core)-(non-core) kets
  const IMSRG_G int *gcore_start, *gcore_loc, *gnc_start, *gnc_loc;
};

// Ket groups of the block-sparse basis transformation: the kets of a channel whose
// orbits come from the same unordered pair of one-body (l, j2, tz2) blocks.
struct XformDev {
  const IMSRG_G int *g_start;   // ngroups + 1: group g holds g_kets[g_start[g] .. g_start[g+1])
  const IMSRG_G int *g_kets;    // channel-local ket indices, ascending within a group
  const IMSRG_G int *g_ch;      // channel of each group
  const IMSRG_G long *g_doff;   // offset of each group's fragments of D
  const IMSRG_G int *c_start;   // channel c's groups are c_start[c] .. c_start[c+1] - 1
  int ngroups, maxm;
};

// Everything one commutator needs: operand buffers, workspaces, flags.
struct PairPtrs {
  const IMSRG_G BasisDev *basis;  // device pointer
  const IMSRG_G double *X, *Y;    // operator buffers (zero | one | two)
  IMSRG_G double *Z;
  IMSRG_G double *Xt, *Yt, *Zbar; // Pandya workspaces
  IMSRG_G double *scratch;        // >= nch + 8 doubles (zero-body partial sums)
  IMSRG_G double *obpart;         // per-call one-body partial sums, nobpart entries
  IMSRG_G double *diag;           // per-call inverse-Pandya diagonal terms, one per ket of every channel (ndiag)
  IMSRG_G double *panel;          // per-call bf16x3 panels of the mixed pp/hh GEMM (2 pk_size doubles)
  IMSRG_G double *c122w;          // per-call comm122 W, two-body layout (tbsize + 8 doubles)
  int hX, hY, hZ;
  unsigned mask;
};

struct PairArg {
  PairPtrs p0;           // used when tab == nullptr
  const IMSRG_G PairPtrs *tab;  // batched: device table
  __device__ __forceinline__ PairPtrs get(int i) const {
    if (tab) return tab[i];  // separate returns keep each load in its own address space
    return p0;
  }
};

// LDS layout of the inverse Pandya kernel, in bytes
struct InvpLds {
  int set, q, z, cls, row, cf, pre, tab, quad, chunk, M;
  __host__ __device__ InvpLds(int nJ, int nt, int norb, int ncls, int nquad, int nchunk) {
    set = 0;                       // int4[nt]: columns in [k0, k1), orbits < k0 of j's and of i's set
    q = set + 16 * nt;             // int4[2 nt]: offset, rows, columns, first entry of cc_cols of the blocks
    z = q + 32 * nt;               // int4[nt]: offset of the first row's elements (low, high), CC channel size
    cls = z + 16 * nt;             // int4[2 ncls]: the classes' kets and J (first ncls) and J' and weights
    row = cls + 32 * ncls;         // long[nJ + 16]: byte offset of the bra's row of the channel 6J + g, or -1
    cf = row + 8 * (nJ + 16);      // int[2 nt + 2]: first chunk of each block, then all elements
    pre = cf + 4 * (2 * nt + 2);   // int[ncls + 1]: first result quad of each class
    tab = (pre + 4 * (ncls + 1) + 15) & ~15;    // ushort2[(nt / 4 + 1) norb4]: column offset and row of (J', orbit)
    quad = tab + (nt + 4) * ((norb + 3) & ~3);  // unsigned[nquad]: class << 20 | J quad << 15 | ket quad
    chunk = quad + 4 * nquad;      // ushort[nchunk]: block of each chunk
    M = (chunk + 2 * nchunk + 15) & ~15;
  }
};

__host__ __device__ inline int ket_index(int norb, int p, int q) { return p * (2 * norb - 1 - p) / 2 + q; }
__host__ __device__ inline int sgn_parity(int x) { return (x & 1) ? -1 : 1; }
__host__ __device__ inline long sixjQ_index(int d1, int d2, int jj1, int jj2, int J3, int jj4, int jj5, int J6) {
  return (((((long)((jj1 - 1) >> 1) * d1 + ((jj2 - 1) >> 1)) * d1 + ((jj4 - 1) >> 1)) * d1 + ((jj5 - 1) >> 1)) * d2 +
          J6) * d2 + J3;
}
__host__ __device__ inline long sixj_index(int d1, int d2, int jj1, int jj2, int J3, int jj4, int jj5, int J6) {
  return (((((long)((jj1 - 1) >> 1) * d1 + ((jj2 - 1) >> 1)) * d2 + J3) * d1 + ((jj4 - 1) >> 1)) * d1 +
          ((jj5 - 1) >> 1)) * d2 + J6;
}

}  // namespace imsrg
