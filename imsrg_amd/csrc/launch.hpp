// launch.hpp -- host-callable launchers of the HIP kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "internal.hpp"

namespace imsrg {

// dense 6j table {jj1 jj2 J3; jj4 jj5 J6} (double-double Racah): `table` in the layout of
// SixJCache_112112, `tableQ` in the sixjQ_index layout as the weights (2 J6 + 1) {6j},
// 0 in place of |6j| < 1e-8
hipError_t launch_sixj_table(double *table, double *tableQ, int d1, int d2, hipStream_t s);

// commutator phases; items are device arrays of int4 work items
// operands, Hermiticities and terms of up to kMax pairs of a batch, into its device
// table (a kernel argument: nothing of the call stays in host memory)
struct PairOps {
  static constexpr int kMax = 64;
  struct {
    const double *X, *Y;
    double *Z;
    int hX, hY, hZ;
    unsigned mask;
  } op[kMax];
  int n;
};
hipError_t launch_set_pairs(PairPtrs *tab, const PairOps &ops, hipStream_t s);

// first launch: zero-body channels (nzero work-groups per pair: the largest channel
// count + 1; nzeros in all), one-body pairs (comm111 + comm121), comm221 partial sums
// and Pandya chunks side by side; maxnch sizes the Pandya chunks' LDS channel table
struct FrontItems {
  const int4 *one, *ob221, *pandya;
  int nzero, nzeros, none, n221, npandya;
  bool xbar_f32;  // Xbar and Ybar in FP32 (the ph GEMM on 128x128 tiles with FP32 products reads them so)
  // small bases: the 64x64 pp/hh tiles and comm122's W items, in the same launch
  const int4 *pphh64, *c122;
  int n64, nc122;
  bool split;  // the Pandya chunks in a launch of their own, after the others (kFrontSplit)
  int blocks() const { return n64 + nc122 + nzeros + none + n221 + npandya; }
};
// mixed64: the pp/hh tiles with FP32 products
hipError_t launch_front(const PairArg &pa, const FrontItems &f, int maxnch, int maxbin, bool mixed64, hipStream_t s);
// Work-groups up to which the first launch takes those as well: one launch, and without
// 128x128 pp/hh tiles no second stream, instead of three launches and four stream events,
// which cost the smallest bases more than their work (emax = 2 FP64 49 -> 28 us, emax = 3
// 50 -> 34, emax = 5 90 -> 87, mixed 71 -> 68, emax = 6 147 -> 140 and 99 -> 93 us).  Where they fill
// the chip they only hold up the main stream: emax = 7 235 -> 239 us, mixed 161 -> 174 us.
constexpr int kFrontSmall = 3500;
// 128x128 pp/hh tiles (two for each CU) above which the first launch of one commutator is two,
// the Pandya chunks after the others: the FP64, FP32 and split FP32 GEMMs beside it take all
// registers of a CU then, and the two launches together wait less for them than one (FP64 emax =
// 9, 747 tiles, O16 1088 -> 1085 us and Ca40 1399 -> 1379, emax = 10 O16 2616 -> 2590 and Ca40 3222 ->
// 3190, emax = 12 14.45 -> 14.3 ms; FP32 emax = 9 927 -> 914, emax = 10 2196 -> 2145; split emax = 10
// 4824 -> 4643).  Not so with fewer tiles (FP64 emax = 8, 393 tiles, O16 469 -> 485 us, Ca40 604 ->
// 638; emax = 7 235 -> 258), beside the bf16x3 GEMM, one work-group per CU (mixed emax = 8 Ca40
// 465 -> 477, emax = 10 O16 1728 -> 1761, Ca40 2200 -> 2202, emax = 12 8.24 -> 8.22 ms), and in
// batches (FP64, 24 pairs at emax = 6 1501 -> 1515 us, 8 at emax = 8 3.43 -> 3.43 ms).  Split products,
// three times the FP32 work per tile: from half as many (emax = 8 Ca40 1032 -> 987 us).
constexpr int kFrontSplit = 512;
// pp/hh SYR2K: items on 128x128 tiles, items64 on 64x64 tiles (disjoint channels);
// under bf16x3 products (kGemmB3) the pack items first write the operand panels
// maxn: the largest channel dimension of the pairs (sizes the kernel's LDS index list)
hipError_t launch_pphh(const PairArg &pa, const int4 *items, int nitems, const int4 *items64, int nitems64,
                       const int4 *pack, int npack, int precision, int maxn, hipStream_t s);
// ph GEMM (head and tail of Zbar) on 128x128 tiles (big) or 64x64 tiles; precision 1
// (FP32 products) stores Zbar in FP32, the others in FP64
hipError_t launch_ph_gemm(const PairArg &pa, const int4 *items, int nitems, int precision, bool big, hipStream_t s);
// lds: DeviceBasis::invp_lds, the largest of the pairs; zbar_f32: Zbar holds FP32 elements
// (written by the precision-1 ph GEMM)
hipError_t launch_invpandya(const PairArg &pa, const int4 *items, int nitems, size_t lds, bool zbar_f32,
                            hipStream_t s);
// last launch: with fold, upper += the inverse-Pandya contributions stored at the
// transposed slots; with c122, Z2 -= W + hZ W^T (comm122ss); then lower triangle
// <- hZ * upper; and Z0 and Z1 from the first launch's partial sums
hipError_t launch_finish(const PairArg &pa, const int4 *items, int nitems, bool fold, bool c122, int npairs,
                         int maxn1pairs, hipStream_t s);
// comm122's W (two-body layout, P.c122w) by column bins; before launch_finish with c122
hipError_t launch_c122_w(const PairArg &pa, const int4 *items, int nitems, int maxbin, hipStream_t s);
hipError_t launch_zero_two(const PairArg &pa, const int4 *items, int nitems, hipStream_t s);

// operator arithmetic
// y = z + a x; z may be y
hipError_t launch_axpy(double *y, const double *z, double a, const double *x, long n, hipStream_t s);
hipError_t launch_scale(double *y, double a, long n, hipStream_t s);
hipError_t launch_fill(double *y, double v, long n, hipStream_t s);  // y[i] = v
// Operator::DoNormalOrdering2 / UndoNormalOrdering of a scalar operator in place
// (sign +1 / -1); n2sq: the squared two-body norm on the device (launch_norm's second
// value): the one-body sum over the holes runs when the norm exceeds 1e-7, the
// (anti-)Hermitian completion of the one-body part always
hipError_t launch_normal_order(const BasisDev *bd, const BasisDev &bh, double *op, int sign, int herm,
                               const double *n2sq, hipStream_t s);
// sums of squares of an operator buffer x into out[0] (one-body) and out[1] (two-body,
// weighted), and in the same pass kAxpy: y = z + a x (z may be y), kCopy: y = x over the whole buffer;
// seq != 0: out and *done are host memory, *done = seq once out holds the sums
enum class NormOp { kSum, kAxpy, kCopy };
hipError_t launch_norm(const BasisDev *bd, const BasisDev &bh, NormOp op, double *y, const double *z, double a,
                       const double *x, double *partials, int maxpart, double *out, unsigned long long *done,
                       unsigned long long seq, hipStream_t s);
// the Hartree-Fock monopoles W[q] = sum_J (2J+1) V~^J_{ia,jb} of quads[q] = (i, a, j, b)
hipError_t launch_hf_mono(const BasisDev *bd, const double *op, const int4 *quads, int nq, double *W,
                          hipStream_t s);
// block-sparse basis transformation (C block diagonal in (l, j2, tz2)): the groups' D
// fragments into Dg, then two passes over items (group, first row; kXfRows rows each; group
// -1: none), T = (V D)^T and out two-body = D^T V D (herm 0: neither Hermitian nor
// anti-Hermitian), and out one-body = C^T O C (through one_tmp)
hipError_t launch_xform_blocks(const BasisDev *bd, const BasisDev &bh, const XformDev &X, const double *C,
                               const double *op, double *out, double *T, double *Dg, double *one_tmp,
                               const int2 *items, int nitems, int herm, hipStream_t s);
// the basis-change matrices D of every channel (two-body layout, tbsize doubles) from
// the one-body basis change C (norb x norb, column-major)
hipError_t launch_hf_D(const BasisDev *bd, const BasisDev &bh, const double *C, double *D, hipStream_t s);
hipError_t launch_fill_random(const BasisDev *bd, const BasisDev &bh, double *op, int herm,
                              unsigned long long seed, hipStream_t s);
hipError_t launch_white(const BasisDev *bd, const BasisDev &bh, const double *H, double *Eta, const int4 *gen_items,
                        int ngen, hipStream_t s);

// met[1] = whether work on `setter` ran while `waiter` was busy (met[0] = 0 beforehand;
// waits at most `ticks` of the 100 MHz clock)
hipError_t launch_meet(int *met, long long ticks, hipStream_t waiter, hipStream_t setter);

// self-test of the MFMA f64 and f32 lane layouts: out[1024] (see imsrg_hip_selftest_mfma)
hipError_t launch_mfma_probe(double *out, hipStream_t s);
// one v_mfma_f32_16x16x32_bf16 on host-given operand slots (a, b: 512 floats, d: 256)
hipError_t launch_mfma_bf16_probe(const float *a, const float *b, float *d, hipStream_t s);

}  // namespace imsrg
