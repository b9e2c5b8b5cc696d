// HIP kernels of the IMSRG(2) scalar-commutator path for gfx950 (CDNA4).
//
//  * k_comm122p, k_comm222ph_scatter, k_pandya: per-element gathers, one
//    thread per output element, 256-element tiles from a task list that
//    spans every channel (grouped) or one channel (plain path);
//    k_comm222ph_chunk: the grouped inverse Pandya by quadruple chunks.
//  * the FP64 MFMA GEMMs live in gemm.hip; k_pppp_sym applies the
//    reference's  W - pm W^T  epilogue of 222_pp_hh to the pppp product.
//  * one-body terms, norms, axpy, generator, mbpt2 and normal ordering.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "gemm_tile.hpp"
#include "kernels.hpp"

namespace imsrg {

// ============================================================ commutator_122
// commutators.f90:283-396.  RES two-body = 1b x 2b part (assigned): for
// every stored element (ab,cd) at J, the sums over the (l,j,tz) block
// partners i of a, b, c, d of f(L)*v(R) - f(R)*v(L), then divided by
// sqrt(1+delta_ab) sqrt(1+delta_cd).
// The partner lists are precomputed per stored pair (a-, b-, c-, d-replaced,
// in that order), so no term performs an index search.

// one partner term: f (from LDS) times the operand elements r = R[o],
// l = L[o], accumulated as sm + fl*vr - fr*vl (row partners) or
// sm - fl*vr + fr*vl (column partners), vr = r * pre * (Rh if the element
// is read from the transposed block), vl = l * pre * (Lh likewise), fl / fr
// times Lh / Rh when the record's one-body element is read transposed.
// Those herm factors and the record's sign are +-1: they combine into one
// sign bit per product, applied to pre = pre_other * (1 or sqrt 2)
// (pa1 / pa2).  lneg / rneg: Lh / Rh < 0.
template <bool ROW>
__device__ __forceinline__ double term122(double sm, const Partner p, double r, double l, const PartnerAddr A,
                                          double pa1, double pa2, const double* s_f, int nf1, int lneg, int rneg) {
  const int code = p.code;
  const int tr = pa_trans(A, (code >> 22) & 3);
  const int fs = (code >> 24) & 1, neg = (code >> 25) & 1;
  const double a = ((code >> 26) & 1) ? pa2 : pa1;
  const int sr = neg ^ (fs & lneg) ^ (tr & rneg);   // sign of the R-operand product
  const int sl = neg ^ (fs & rneg) ^ (tr & lneg);   // sign of the L-operand product
  const double cr = (sr ^ (ROW ? 0 : 1)) ? -a : a, cl = (sl ^ (ROW ? 1 : 0)) ? -a : a;
  sm = fma(s_f[p.fk] * cr, r, sm);
  return fma(s_f[nf1 + p.fk] * cl, l, sm);
}

// the n partner terms of one list, record k at part[k * ps], IMSRG_122_UNROLL
// records and their operand loads in flight at a time; the terms are added
// in list order
#ifndef IMSRG_122_UNROLL
#define IMSRG_122_UNROLL 2
#endif
template <bool ROW>
__device__ __forceinline__ double sum122(double sm, const Partner* part, i64 ps, int n, const PartnerAddr A,
                                         double pa1, double pa2, const double* s_f, int nf1, const double* L,
                                         int lneg, const double* R, int rneg) {
  constexpr int U = IMSRG_122_UNROLL;
  int x = 0;
  for (; x + U - 1 < n; x += U) {
    Partner p[U];
    double r[U], l[U];
#pragma unroll
    for (int u = 0; u < U; ++u) p[u] = part[(x + u) * ps];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const i64 o = pa_off(A, (p[u].code >> 22) & 3, p[u].code & 0x3fffff);
      r[u] = R[o];
      l[u] = L[o];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) sm = term122<ROW>(sm, p[u], r[u], l[u], A, pa1, pa2, s_f, nf1, lneg, rneg);
  }
  for (; x < n; ++x) {
    const Partner p = part[x * ps];
    const i64 o = pa_off(A, (p.code >> 22) & 3, p.code & 0x3fffff);
    sm = term122<ROW>(sm, p, R[o], L[o], A, pa1, pa2, s_f, nf1, lneg, rneg);
  }
  return sm;
}

__device__ __forceinline__ void d_comm122p(DevBasis B, const SegTask* tasks, const Partner* part,
                                           const Partner* partT, int pstride, const int* rowp, const int* colp,
                                           const int* f1off, int nf1, const double* L, int Lh, const double* R,
                                           int Rh, double* RES, int RESh, int mirror, int bx, int nbx,
                                           double* s_f) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  RES += (i64)inst * B.oplen;
  // the one-body elements the partner terms read, L then R, staged once
  for (int k = threadIdx.x; k < nf1; k += blockDim.x) {
    const int o = f1off[k];
    s_f[k] = L[o];
    s_f[nf1 + k] = R[o];
  }
  __syncthreads();
  const SegTask t = tasks[xcd_contig(bx, nbx)];   // neighbouring tiles share partner rows
  const i64 e = (i64)t.start + threadIdx.x;
  if (e >= t.cnt) return;
  const int q = t.q, g = t.g;
  const int rc = row_cls(g), cc = col_cls(g);
  const int n1 = B.dims[q * 3 + rc];
  const bool sq = is_square(g);
  int IX, JX;
  if (sq) upper_decode(e, IX, JX);
  else { IX = (int)(e % n1); JX = (int)(e / n1); }
  const i64 gr = B.pairoff[q * 3 + rc] + IX, gc = B.pairoff[q * 3 + cc] + JX;
  int a, b, c, d;
  unpack(B.pairs[gr], a, b);
  unpack(B.pairs[gc], c, d);
  const double pre_ab = (a == b) ? 1.4142135623730951 : 1.0;
  const double pre_cd = (c == d) ? 1.4142135623730951 : 1.0;
  PartnerAddr AR, AC;
  partner_addr(B.goff + q * 6, B.dims + q * 3, rc, cc, IX, JX, AR, AC);   // uniform (scalar) loads
  double sm = 0.0;
  const int lneg = Lh < 0, rneg = Rh < 0;
  sm = sum122<true>(sm, partT + gr, pstride, rowp[gr + 1] - rowp[gr], AR, pre_cd, pre_cd * 1.4142135623730951, s_f,
                    nf1, L, lneg, R, rneg);
  // column partners: when every active lane of the wave holds an element of
  // one column pair (the common case), the list is read through the scalar
  // cache instead of once per lane
  const int gc0 = __builtin_amdgcn_readfirstlane((int)gc);
  if (__all((int)gc == gc0)) {
    const int x0 = colp[gc0], nx = colp[gc0 + 1] - x0;
    sm = sum122<false>(sm, part + x0, 1, nx, AC, pre_ab, pre_ab * 1.4142135623730951, s_f, nf1, L, lneg, R, rneg);
  } else {
    sm = sum122<false>(sm, part + colp[gc], 1, colp[gc + 1] - colp[gc], AC, pre_ab, pre_ab * 1.4142135623730951, s_f,
                       nf1, L, lneg, R, rneg);
  }
  sm = sm / sqrt(1.0 + (a == b ? 1.0 : 0.0)) / sqrt(1.0 + (c == d ? 1.0 : 0.0));
  const i64 base = B.goff[q * 6 + g];
  RES[base + IX + (i64)JX * n1] = sm;
  if (sq && mirror) RES[base + JX + (i64)IX * n1] = sm * RESh;
}

__global__ __launch_bounds__(256) void k_comm122p(DevBasis B, const SegTask* tasks, const Partner* part,
                                                  const Partner* partT, int pstride, const int* rowp,
                                                  const int* colp, const int* f1off, int nf1, const double* L,
                                                  int Lh, const double* R, int Rh, double* RES, int RESh,
                                                  int mirror) {
  extern __shared__ double s_f[];
  d_comm122p(B, tasks, part, partT, pstride, rowp, colp, f1off, nf1, L, Lh, R, Rh, RES, RESh, mirror, blockIdx.x, gridDim.x, s_f);
}

void launch_comm122p(const DevBasis& B, const SegTask* t, int nt, const Partner* part, const Partner* partT,
                     int pstride, const int* rowp, const int* colp, const int* f1off, int nf1, const double* L, int Lh,
                     const double* R, int Rh, double* RES, int RESh, hipStream_t s, int mirror) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_comm122p, dim3(nt, B.ninst), dim3(kTile), 2 * nf1 * sizeof(double), s, B, t, part, partT,
                     pstride, rowp, colp, f1off, nf1, L, Lh, R, Rh, RES, RESh, mirror);
}

// ---------------------------------------------- commutator_122 by closed tiles
// One workgroup per tile (row group x column slab, see T122Plan) of one
// channel.  The tile of both operands is staged in LDS as full-matrix elements
// M(r, c) (herm applied to elements stored transposed), so each stored
// element is read from memory once, along contiguous runs of the ordered row
// entries; the partner sums
//   RES(r, c) = sum_k FL(r, k) R(k, c) - FR(r, k) L(k, c)
//             - sum_k R(r, k) GL(k, c) - L(r, k) GR(k, c)
// then read LDS only.  Lanes hold the rows (their records' coefficients in
// registers), waves take the columns (their records broadcast from LDS).
// Tiles cover every unordered pair of groups once: off the diagonal the
// elements of (column, row) follow from RES(c, r) = -Lh Rh RES(r, c) and are
// written through LDS along the columns, so both orientations are stored in
// contiguous runs.  mirror = 0: only the upper triangles of the square blocks.
// mirror = 1: the lower triangles as well, always RESh times the upper element.
// A diagonal tile sums both, in another order, so it stores its upper ones twice,
// the image in scattered single elements: eMax 6 16.4 us, 7 34.0, 8 70.3 (with its
// own lower sums, in runs, 16.5, 33.9, 69.3; the image through LDS 17.8, 36.4, 72.7).
// The list kernel above is bound by the address path (about 42 vector loads an
// element); here an element costs two loads, one store and about 30 LDS reads.
// What bounds it now is the chain of a tile (entries, records, coefficients,
// elements, sums: waves wait 56 % of their cycles at four a SIMD) and, at eMax
// 10, HBM: 850 MB in 404 us.  Upper triangles, eMax 6 / 8 / 10: 15.3 / 64 / 404
// us against 17.5 / 128 / 892 us by lists.  Tried and slower: several slabs a
// workgroup (the addresses kept across slabs spill), one wave's own copy of
// the row coefficients (12 dependent loads a lane), the columns as the outer
// loop of the row sums (a branch per record and column).
// coefficient of a record for one operand's one-body element f: its sign and
// sqrt 2 factor, and the herm factor of an element read transposed
__device__ __forceinline__ double t122_coef(int rec, double f, int neg_tr) {
  const int k = (rec >> 19) & 3;
  const double a = k == 0 ? f : f * (k == 1 ? 1.4142135623730951 : 0.70710678118654757);
  return (((rec >> 18) & 1) ^ (((rec >> 17) & 1) & neg_tr)) ? -a : a;
}

// MAXR: records of a row held in registers; NJ: columns of a wave (4 NJ >= slab)
template <int MAXR, int NJ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NJ <= 8 ? 4 : 3))) void k_comm122t(
    DevBasis B, T122Plan P, const T122Task* tasks, const double* L, int Lh, const double* R, int Rh, double* RES,
    int RESh, int mirror) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  RES += (i64)inst * B.oplen;
  // (row r, column c) of the tiles at c * LD + r: compile-time strides, so the
  // columns of a wave are immediate offsets of one address per record; the
  // padding row kT122Rows holds zeros, read by the lanes with fewer records
  constexpr int LD = kT122Rows + 1, NC = 4 * NJ;
  static_assert(2 * MAXR * kT122Rows <= 2 * NC * LD, "the row coefficients pass through the tiles' LDS");
  __shared__ double tile[2 * NC * LD];
  __shared__ double cf[2 * NC * MAXR];   // column coefficients (gL, gR) of record k of column c
  __shared__ int cl[NC * MAXR];          // their column offsets in the tile
  double* const tL = tile;
  double* const tR = tile + NC * LD;
  const T122Task t = tasks[xcd_contig(blockIdx.x, gridDim.x)];   // neighbouring tiles share lines
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lneg = Lh < 0, rneg = Rh < 0;
  const int nrow = t.nrow;
  const i64* go = B.goff + t.q * 6;
  const int d0 = B.dims[t.q * 3], d1 = B.dims[t.q * 3 + 1], d2 = B.dims[t.q * 3 + 2];
  const i64 g0 = go[0], g11 = go[3], g22 = go[4], x12 = go[5] - go[3];
  const bool rok = lane < nrow;
  const int re = rok ? P.rent[t.row0 + lane] : 0;
  const int nr = rok ? P.rcnt[t.row0 + lane] : 0;
  const int rcls = re >> 28, ridx = re & 0xfffffff;
  const int ldr = pick3(rcls, d0, d1, d2);
  // Stored position of (row, column of class cc and index ic), row class <=
  // cc: the blocks of row class pp are one matrix of d0 rows over all columns
  // (p0 = the column's place there); class ph has two blocks, hh one.
  const i64 rbase = (rcls == 0 ? g0 : (rcls == 1 ? g11 : g22)) + ridx;
  auto at = [&](int cc, int ic, int p0) -> i64 {
    return rbase + (i64)(rcls == 0 ? p0 : ic) * ldr + (rcls == 1 && cc == 2 ? x12 : 0);
  };
  const int np = __popcll(__ballot(rok && rcls == 0));   // rows of class pp (the entries are ordered by class)
  int nmax = nr;   // most records of a row
  for (int o = 32; o > 0; o >>= 1) nmax = max(nmax, __shfl_xor(nmax, o, 64));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  const int hnat = -Lh * Rh;
  double fl[MAXR], fr[MAXR];
  int rl[MAXR];
  const int ncol = t.ncol;
  const bool cok = lane < ncol;
  // column entries and record counts, column c in lane c of every wave
  const int ce_l = cok ? P.cent[t.col0 + lane] : 0;
  const int cn_l = cok ? P.ccnt[t.col0 + lane] : 0;
  const int ccls_l = ce_l >> 28, cidx_l = ce_l & 0xfffffff;
  const int p0_l = cidx_l + pick3(ccls_l, 0, d0, d0 + d1);
  // elements stored as (r, c), lanes along the rows, into registers
  double pl[NJ], pr[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int c = wave + 4 * j;
    pl[j] = pr[j] = 0.0;
    if (c < ncol) {
      const int ce = __builtin_amdgcn_readlane(ce_l, c), p0 = __builtin_amdgcn_readlane(p0_l, c);
      if (rok && rcls <= (ce >> 28)) {
        const i64 o = at(ce >> 28, ce & 0xfffffff, p0);
        pl[j] = L[o];
        pr[j] = R[o];
      }
    }
  }
  // column coefficients
  for (int x = tid; x < ncol * MAXR; x += 256) {
    const int c = x / MAXR, k = x - c * MAXR;
    if (k < P.ccnt[t.col0 + c]) {
      const int2 rec = P.crec[(i64)k * P.ncols + t.col0 + c];
      cf[2 * x] = t122_coef(rec.x, L[rec.y], lneg);
      cf[2 * x + 1] = t122_coef(rec.x, R[rec.y], rneg);
      cl[x] = (rec.x & 63) * LD;
    }
  }
  // row coefficients, formed once by the workgroup and kept in every
  // wave's registers
  {
    for (int x = tid; x < nmax * kT122Rows; x += 256) {
      const int r = x & (kT122Rows - 1), k = x / kT122Rows;   // this lane's own row
      double vl = 0.0, vr = 0.0;
      if (k < nr) {
        const int2 rec = P.rrec[(i64)k * P.nrows + t.row0 + r];
        vl = t122_coef(rec.x, L[rec.y], lneg);
        vr = t122_coef(rec.x, R[rec.y], rneg);
      }
      tile[2 * x] = vl;
      tile[2 * x + 1] = vr;
    }
#pragma unroll
    for (int k = 0; k < MAXR; ++k)
      rl[k] = wave * LD + (k < nr ? (P.rrec[(i64)k * P.nrows + t.row0 + lane].x & 63) : kT122Rows);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < MAXR; ++k)
      if (k < nmax) {
        fl[k] = tile[2 * (k * kT122Rows + lane)];
        fr[k] = tile[2 * (k * kT122Rows + lane) + 1];
      }
    __syncthreads();
  }
  if (tid < NC) tL[tid * LD + kT122Rows] = tR[tid * LD + kT122Rows] = 0.0;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int c = wave + 4 * j;
    if (c < ncol && rok && rcls <= (__builtin_amdgcn_readlane(ce_l, c) >> 28)) {
      tL[c * LD + lane] = pl[j];
      tR[c * LD + lane] = pr[j];
    }
  }
  // elements stored as (c, r), class of c below the class of r: lanes along
  // the columns
  const i64 cbase = (ccls_l == 0 ? g0 : (ccls_l == 1 ? g11 : g22)) + cidx_l;
  const int ldc = pick3(ccls_l, d0, d1, d2);
  auto atc = [&](int kr, int ir) -> i64 {
    return cbase + (i64)(ccls_l == 0 ? ir + pick3(kr, 0, d0, d0 + d1) : ir) * ldc + (ccls_l == 1 && kr == 2 ? x12 : 0);
  };
#pragma unroll 4
  for (int r = np + wave; r < nrow; r += 4) {
    const int er = __builtin_amdgcn_readlane(re, r);
    const int kr = er >> 28;
    if (cok && ccls_l < kr) {
      const i64 o = atc(kr, er & 0xfffffff);
      tL[lane * LD + r] = Lh * L[o];
      tR[lane * LD + r] = Rh * R[o];
    }
  }
  __syncthreads();
  // this lane's outputs of columns wave, wave + 4, ... (those past the slab
  // sum whatever the tile holds and are not stored)
  double val[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) val[j] = 0.0;
#pragma unroll
  for (int k = 0; k < MAXR; ++k)
    if (k < nmax) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        val[j] = fma(fl[k], tR[rl[k] + 4 * j * LD], val[j]);
        val[j] = fma(-fr[k], tL[rl[k] + 4 * j * LD], val[j]);
      }
    }
  const int row = rok ? lane : kT122Rows;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int c = wave + 4 * j;
    if (c < ncol) {
      const int nk = __builtin_amdgcn_readlane(cn_l, c);
      const int* clc = cl + c * MAXR;
      const double* cfc = cf + 2 * c * MAXR;
#pragma unroll 2
      for (int k = 0; k < nk; ++k) {
        const int o = clc[k] + row;
        val[j] = fma(-cfc[2 * k], tR[o], val[j]);
        val[j] = fma(cfc[2 * k + 1], tL[o], val[j]);
      }
    }
  }
  // outputs stored as (r, c)
  const bool lower = mirror && !t.diag;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int c = wave + 4 * j;
    if (c < ncol) {
      const int ce = __builtin_amdgcn_readlane(ce_l, c), p0 = __builtin_amdgcn_readlane(p0_l, c);
      const int cc = ce >> 28, ic = ce & 0xfffffff;
      // kept: every class pair below the diagonal, the upper triangle and,
      // with mirror, the lower one of the square blocks
      if (rok && (rcls < cc || (rcls == cc && (lower || ridx <= ic))))
        RES[at(cc, ic, p0)] =
            rcls < cc || ridx < ic ? val[j] : (ridx == ic ? (mirror ? val[j] * RESh : val[j]) : val[j] * (hnat * RESh));
    }
  }
  if (t.diag) {
    if (!mirror) return;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int c = wave + 4 * j;
      if (c < ncol) {   // row ic, column ridx
        const int ce = __builtin_amdgcn_readlane(ce_l, c), p0 = __builtin_amdgcn_readlane(p0_l, c);
        const int cc = ce >> 28, ic = ce & 0xfffffff;
        if (rok && rcls == cc && ridx < ic) RES[at(cc, ridx, p0 - ic + ridx) + (ic - ridx)] = val[j] * RESh;
      }
    }
    return;
  }
  // the other orientation, through LDS: lanes along the columns
  __syncthreads();
  {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int c = wave + 4 * j;
      if (c < ncol && rok) tL[c * LD + lane] = val[j];
    }
    __syncthreads();
#pragma unroll 2
    for (int r = wave; r < nrow; r += 4) {
      const int er = __builtin_amdgcn_readlane(re, r);
      const int kr = er >> 28, ir = er & 0xfffffff;
      if (cok && (ccls_l < kr || (ccls_l == kr && (mirror || cidx_l < ir)))) {
        const double v = tL[lane * LD + r];
        RES[atc(kr, ir)] = v * (ccls_l < kr || cidx_l < ir ? hnat : RESh);
      }
    }
  }
}

void launch_comm122t(const DevBasis& B, const T122Plan& P, const T122Task* t, int nt, const double* L, int Lh,
                     const double* R, int Rh, double* RES, int RESh, hipStream_t s, int mirror) {
  if (nt <= 0) return;
  const dim3 g(nt, B.ninst), w(256);
#define IMSRG_122T(MR, NJ) \
  hipLaunchKernelGGL((k_comm122t<MR, NJ>), g, w, 0, s, B, P, t, L, Lh, R, Rh, RES, RESh, mirror)
  // blocks of n orbits have n^2 columns and 2 n records: n <= 4, 5, 6, 7
  if (P.maxrec <= 8 && P.maxcol <= 16) IMSRG_122T(8, 4);
  else if (P.maxrec <= 10 && P.maxcol <= 32) IMSRG_122T(10, 8);
  else if (P.maxrec <= 12 && P.maxcol <= 40) IMSRG_122T(12, 10);
  else IMSRG_122T(16, 14);
#undef IMSRG_122T
}

// ================================================== commutator_222_ph scatter
// commutators.f90:804-923.  Every J' term of the reference reads WCC and
// its transpose only in the combination
//     W'(x,y) = Lh W(x,y) - Rh W(y,x),    W = LCC RCC^T,
// inside:  (W(gik,rjl) + ph W(gjl,rik)) Lh - (ph W(rik,gjl) + W(rjl,gik)) Rh
//        =  W'(gik,rjl) + ph W'(gjl,rik)
// outside: W'(gil,rjk) + ph W'(gjk,ril).
// W' satisfies W'(y,x) = -Lh Rh W'(x,y), so the GEMM stores its upper
// triangle only and the scatter reads the element (min, max).  (Storing
// both triangles, for reads along columns only, costs the GEMM more in
// transposed stores than it saves here.)

// sixj for arguments whose four triangle conditions hold by construction
// (the J' ranges below), so the table read is unconditional
__device__ __forceinline__ double sixj_tri(const DevBasis& B, int j1, int j2, int j3, int j4, int j5, int j6) {
  const int nh = B.nh6;
  const i64 idx = (((((i64)(j1 >> 1) * nh + (j2 >> 1)) * nh + (j4 >> 1)) * nh + (j5 >> 1)) * B.nJ6 + (j6 >> 1)) *
                      B.nJ6 + (j3 >> 1);
  return B.six[idx];
}

// One recoupling's sum over J' (jmin..jmax step 2), added onto sm:
//   inside:  - (-1)^((jl+jk+J)/2) (W'(gik,rjl) + phase W'(gjl,rik)) {ji jj J; jl jk J'}
//   outside: + (W'(gil,rjk) + phase W'(gjk,ril)) {ji jj J; jk jl J'}
// ph_pair gives the W' combination of one J' term.
// JFAST: the row tables read with J' fastest (rmap; the grouped form runs
// the consecutive J' terms of one quadruple in neighbouring lanes, which
// then read neighbouring entries), else with J' slowest (rmapJ / rmapJT;
// the per-channel form runs neighbouring i in neighbouring lanes)
template <bool INSIDE, bool JFAST>
__device__ __forceinline__ double ph_pair(const DevBasis& B, const i64* wcoff, const int* rlen, const double* WCC,
                                          double mpm, int phase, int i, int j, int k, int l, int JP, int Tz, int PAR) {
  // inside reads rows (k,i) / cols (j,l); outside rows (l,i) / cols (j,k).
  // 32-bit element offsets from uniform bases (WCC holds < 2^32 doubles,
  // checked at plan time)
  const int N = B.N, JTM = B.JTM, nJ = B.nJ, h = JP >> 1;
  const int a = INSIDE ? k : l, c = INSIDE ? l : k;
  const int qx = h + Tz * (JTM + 1) + 2 * PAR * (JTM + 1);
  const unsigned wo = (unsigned)wcoff[qx], rr = (unsigned)rlen[qx];
  unsigned x1, y1, x2, y2;
  if (JFAST) {
    x1 = B.rmap[(a * N + i) * nJ + h];   // gik | gil
    y1 = B.rmap[(j * N + c) * nJ + h];   // rjl | rjk
    x2 = B.rmap[(i * N + a) * nJ + h];   // rik | ril
    y2 = B.rmap[(c * N + j) * nJ + h];   // gjl | gjk
  } else {
    const unsigned t = (unsigned)h * (unsigned)(N * N);
    x1 = B.rmapJ[t + a * N + i];
    y1 = B.rmapJ[t + j * N + c];
    x2 = B.rmapJT[t + a * N + i];
    y2 = B.rmapJ[t + c * N + j];
  }
  // W'(x1, y1) + phase W'(y2, x2), each read from the upper triangle
  const double A1 = x1 <= y1 ? WCC[wo + x1 + y1 * rr] : mpm * WCC[wo + y1 + x1 * rr];
  const double A2 = y2 <= x2 ? WCC[wo + y2 + x2 * rr] : mpm * WCC[wo + x2 + y2 * rr];
  return A1 + phase * A2;
}

template <bool INSIDE>
__device__ __forceinline__ double ph_jsum(const DevBasis& B, const double* WCC, double mpm, int i, int j, int k, int l,
                                          int Jtot, int jmin, int jmax, int phase, int Tz, int PAR, double sm) {
  const int ji = B.jj[i], jj = B.jj[j], jk = B.jj[k], jl = B.jj[l];
  const double sg = INSIDE ? -(double)m1pow((jl + jk + Jtot) / 2) : 1.0;
  for (int JP = jmin; JP <= jmax; JP += 2) {
    const double v = ph_pair<INSIDE, false>(B, B.wcoff, B.rlen, WCC, mpm, phase, i, j, k, l, JP, Tz, PAR);
    sm = sm + sg * v * (INSIDE ? sixj_tri(B, ji, jj, Jtot, jl, jk, JP) : sixj_tri(B, ji, jj, Jtot, jk, jl, JP));
  }
  return sm;
}

__device__ __forceinline__ void ph_element(const DevBasis& B, const double* WCC, int Lh, int Rh, double* RES,
                                           int RESh, int q, int g, int IX, int JX, int i, int j, int k, int l,
                                           bool mirror = true) {
  const int n1 = brows(B, q, g);
  const bool sq = is_square(g);
  const double pre = (i == j) ? IMSRG_INV_SQRT2_REF : 1.0;
  const double pre2 = (k == l) ? IMSRG_INV_SQRT2_REF : 1.0;
  const double mpm = -(double)(Lh * Rh);
  const int Jtot = B.chJ[q];
  const int ji = B.jj[i], jj = B.jj[j], jk = B.jj[k], jl = B.jj[l];
  const int li = B.ll[i], lj = B.ll[j], lk = B.ll[k], ll = B.ll[l];
  const int ti = B.tz[i], tj = B.tz[j], tk = B.tz[k], tl = B.tz[l];
  const int phase = m1pow((ji + jj + jk + jl) / 2);
  double sm = 0.0;
  // "inside" recoupling
  int Tz = abs(ti - tk) / 2;
  if (abs(tl - tj) != Tz * 2) return;
  int PAR = (li + lk) % 2;
  if ((ll + lj) % 2 != PAR) return;
  sm = ph_jsum<true>(B, WCC, mpm, i, j, k, l, Jtot, max(abs(jj - jl), abs(ji - jk)),
                                min(jj + jl, ji + jk), phase, Tz, PAR, sm);
  // "outside" recoupling
  Tz = abs(ti - tl) / 2;
  if (abs(tk - tj) != Tz * 2) return;
  PAR = (li + ll) % 2;
  if ((lk + lj) % 2 != PAR) return;
  sm = ph_jsum<false>(B, WCC, mpm, i, j, k, l, Jtot, max(abs(ji - jl), abs(jj - jk)),
                                 min(ji + jl, jj + jk), phase, Tz, PAR, sm);
  double* X = RES + B.goff[q * 6 + g];
  const i64 o = IX + (i64)JX * n1;
  X[o] = X[o] + sm * pre * pre2;
  if (sq && mirror) X[JX + (i64)IX * n1] = X[o] * RESh;
}

// per-channel form: segment tiles of one channel (plain path)
__global__ __launch_bounds__(256) void k_comm222ph_scatter(DevBasis B, const SegTask* tasks, const double* WCC,
                                                           int Lh, int Rh, double* RES, int RESh) {
  int inst;
  if (!batch_inst(B, inst)) return;
  WCC += (i64)inst * B.wclen;
  RES += (i64)inst * B.oplen;
  const SegTask t = tasks[blockIdx.x];
  const i64 e = (i64)t.start + threadIdx.x;
  if (e >= t.cnt) return;
  const int q = t.q, g = t.g;
  const int n1 = brows(B, q, g);
  int IX, JX;
  if (is_square(g)) upper_decode(e, IX, JX);
  else { IX = (int)(e % n1); JX = (int)(e / n1); }
  int i, j, k, l;
  unpack(B.pairs[B.pairoff[q * 3 + row_cls(g)] + IX], i, j);
  unpack(B.pairs[B.pairoff[q * 3 + col_cls(g)] + JX], k, l);
  ph_element(B, WCC, Lh, Rh, RES, RESh, q, g, IX, JX, i, j, k, l);
}

void launch_comm222ph_scatter(const DevBasis& B, const SegTask* t, int nt, const double* W, int Lh, int Rh,
                              double* RES, int RESh, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_comm222ph_scatter, dim3(nt, B.ninst), dim3(kTile), 0, s, B, t, W, Lh, Rh, RES, RESh);
}

// J' ranges of the two recouplings of quadruple (i,j,k,l) (empty when
// jmin > jmax); ok = false when an isospin / parity check fails, in which
// case the element receives nothing (as in ph_element)
struct PhRanges { int jin, nin, jout, nout; bool ok; };
__device__ __forceinline__ PhRanges ph_ranges(const DevBasis& B, int i, int j, int k, int l) {
  PhRanges r{0, 0, 0, 0, false};
  const int ji = B.jj[i], jj = B.jj[j], jk = B.jj[k], jl = B.jj[l];
  const int li = B.ll[i], lj = B.ll[j], lk = B.ll[k], ll = B.ll[l];
  const int ti = B.tz[i], tj = B.tz[j], tk = B.tz[k], tl = B.tz[l];
  if (abs(tl - tj) != abs(ti - tk) || (ll + lj) % 2 != (li + lk) % 2) return r;
  if (abs(tk - tj) != abs(ti - tl) || (lk + lj) % 2 != (li + ll) % 2) return r;
  r.ok = true;
  r.jin = max(abs(jj - jl), abs(ji - jk));
  r.nin = max(0, (min(jj + jl, ji + jk) - r.jin) / 2 + 1);
  r.jout = max(abs(ji - jl), abs(jj - jk));
  r.nout = max(0, (min(ji + jl, jj + jk) - r.jout) / 2 + 1);
  return r;
}

// largest x in [0, n) with a[x] <= t (a ascending, a[0] <= t)
__device__ __forceinline__ int lds_floor(const int* a, int n, int t) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// grouped form by quadruple chunks.  Phase 1: one thread per J' term of
// the chunk's quadruples loads its two W' values (index tables, then W')
// into LDS; phase 2: one thread per output (quadruple, J) sums its
// quadruple's terms from LDS with the 6j weights, in the order ph_element
// adds them (same result bits).  Each W' term is fetched once per
// quadruple instead of once per (quadruple, J).
struct PhChunkLds {
  int ijkl[kPhChunkItems], loff[kPhChunkItems], ioff[kPhChunkItems];
  int jin[kPhChunkItems], nin[kPhChunkItems], jout[kPhChunkItems];
  // per quadruple, from the orbit tables once: 2j of i, j, k, l (8 bits
  // each), and the recoupling / output data (phase, Tz and parity of the
  // inside and outside recouplings, the output channel's Tz / parity part,
  // block g and the two (a,a) factors)
  int jq[kPhChunkItems], meta[kPhChunkItems];
  double val[kPhChunkLanes];
  i64 wcoff[kPhMaxCC];
  int rlen[kPhMaxCC];
};
__device__ __forceinline__ void d_comm222ph_chunk(const DevBasis& B, const PhChunk* chunks, const int* fq,
                                                  const int* fql, const int* fqi, const QuadItem* items,
                                                  const double* WCC, int Lh, int Rh, double* RES, int RESh, int mirror,
                                                  int bx, int nbx, PhChunkLds& S) {
  int inst;
  if (!batch_inst(B, inst)) return;
  WCC += (i64)inst * B.wclen;
  RES += (i64)inst * B.oplen;
  int *s_ijkl = S.ijkl, *s_loff = S.loff, *s_ioff = S.ioff, *s_jin = S.jin, *s_nin = S.nin, *s_jout = S.jout;
  int *s_jq = S.jq, *s_meta = S.meta, *s_rlen = S.rlen;
  double* s_val = S.val;
  i64* s_wcoff = S.wcoff;
  const PhChunk c = chunks[xcd_contig(bx, nbx)];   // neighbouring chunks share W' lines
  const int tid = threadIdx.x;
  const double mpm = -(double)(Lh * Rh);
  for (int x = tid; x < B.ncc; x += blockDim.x) {   // cross-coupled block offsets and row counts
    s_wcoff[x] = B.wcoff[x];
    s_rlen[x] = B.rlen[x];
  }
  if (tid < c.nq) {
    const int u = fq[c.q0 + tid];
    const int i = u & 255, j = (u >> 8) & 255, k = (u >> 16) & 255, l = (u >> 24) & 255;
    const PhRanges r = ph_ranges(B, i, j, k, l);
    s_ijkl[tid] = u;
    s_loff[tid] = fql[c.q0 + tid];
    s_ioff[tid] = fqi[c.q0 + tid] - c.item0;
    s_jin[tid] = r.jin;
    s_nin[tid] = r.ok ? r.nin : 0;
    s_jout[tid] = r.ok ? r.jout : -1;   // -1: no contribution at all
    const int ji = B.jj[i], jj = B.jj[j], jk = B.jj[k], jl = B.jj[l];
    const int ti = B.tz[i], tj = B.tz[j], tk = B.tz[k], tl = B.tz[l];
    const int li = B.ll[i], lj = B.ll[j], lk = B.ll[k], ll = B.ll[l];
    const int rc = B.con[i] + B.con[j], cc = B.con[k] + B.con[l];
    const int g = (rc == 0) ? cc : (rc == 1 ? (cc == 1 ? 3 : 5) : 4);
    s_jq[tid] = ji | (jj << 8) | (jk << 16) | (jl << 24);
    // bit 0: phase (-1)^((ji+jj+jk+jl)/2) < 0; 1: Tz in; 2: parity in;
    // 3: Tz out; 4: parity out; 5-7: output block g; 8: i == j; 9: k == l;
    // 10+: the output channel's 2 (Tz + 1) + P
    s_meta[tid] = (((ji + jj + jk + jl) / 2) & 1) | ((abs(ti - tk) / 2) << 1) | (((li + lk) & 1) << 2) |
                  ((abs(ti - tl) / 2) << 3) | (((li + ll) & 1) << 4) | (g << 5) | ((i == j) << 8) |
                  ((k == l) << 9) | ((2 * ((ti + tj) / 2 + 1) + ((li + lj) & 1)) << 10);
  }
  __syncthreads();
  for (int t = tid; t < c.nlanes; t += blockDim.x) {
    const int q = lds_floor(s_loff, c.nq, t);
    const int u = s_ijkl[q], m = s_meta[q];
    const int i = u & 255, j = (u >> 8) & 255, k = (u >> 16) & 255, l = (u >> 24) & 255;
    const int r = t - s_loff[q];
    const int phase = (m & 1) ? -1 : 1;
    double v;
    if (r < s_nin[q])
      v = ph_pair<true, true>(B, s_wcoff, s_rlen, WCC, mpm, phase, i, j, k, l, s_jin[q] + 2 * r, (m >> 1) & 1,
                        (m >> 2) & 1);
    else
      v = ph_pair<false, true>(B, s_wcoff, s_rlen, WCC, mpm, phase, i, j, k, l, s_jout[q] + 2 * (r - s_nin[q]),
                         (m >> 3) & 1, (m >> 4) & 1);
    s_val[t] = v;
  }
  __syncthreads();
  if (tid >= c.nitems) return;
  const int q = lds_floor(s_ioff, c.nq, tid);
  if (s_jout[q] < 0) return;
  const QuadItem it = items[c.item0 + tid];
  const int u = it.ijkl;
  const int i = u & 255, j = (u >> 8) & 255, k = (u >> 16) & 255, l = (u >> 24) & 255;
  const int J = it.J;
  const int jq = s_jq[q], m = s_meta[q];
  const int ji = jq & 255, jj = (jq >> 8) & 255, jk = (jq >> 16) & 255, jl = (jq >> 24) & 255;
  const double* v = s_val + s_loff[q];
  const int nin = s_nin[q], jin = s_jin[q], jout = s_jout[q];
  const int nout = (q + 1 < c.nq ? s_loff[q + 1] : c.nlanes) - s_loff[q] - nin;
  double sm = 0.0;
  const double sg = -(double)m1pow((jl + jk + J) / 2);
  for (int r = 0; r < nin; ++r) sm = sm + sg * v[r] * sixj_tri(B, ji, jj, J, jl, jk, jin + 2 * r);
  for (int r = 0; r < nout; ++r) sm = sm + 1.0 * v[nin + r] * sixj_tri(B, ji, jj, J, jk, jl, jout + 2 * r);
  // output position: channel from (J, Tz, parity), block from the pair classes
  const int qc = 3 * J + (m >> 10);
  const int g = (m >> 5) & 7;
  const int IX = B.xmap[((i64)i * B.N + j) * B.nJ + (J >> 1)];
  const int JX = B.xmap[((i64)k * B.N + l) * B.nJ + (J >> 1)];
  const int n1 = brows(B, qc, g);
  const double pre = ((m >> 8) & 1) ? IMSRG_INV_SQRT2_REF : 1.0;
  const double pre2 = ((m >> 9) & 1) ? IMSRG_INV_SQRT2_REF : 1.0;
  double* X = RES + B.goff[qc * 6 + g];
  const i64 o = IX + (i64)JX * n1;
  X[o] = X[o] + sm * pre * pre2;
  if (is_square(g) && mirror) X[JX + (i64)IX * n1] = X[o] * RESh;
}
__global__ __launch_bounds__(256) void k_comm222ph_chunk(DevBasis B, const PhChunk* chunks, const int* fq,
                                                         const int* fql, const int* fqi, const QuadItem* items,
                                                         const double* WCC, int Lh, int Rh, double* RES, int RESh,
                                                         int mirror) {
  __shared__ PhChunkLds S;
  d_comm222ph_chunk(B, chunks, fq, fql, fqi, items, WCC, Lh, Rh, RES, RESh, mirror, blockIdx.x, gridDim.x, S);
}

void launch_comm222ph_chunk(const DevBasis& B, const PhChunk* ch, int nch, const int* fq, const int* fql,
                            const int* fqi, const QuadItem* items, const double* W, int Lh, int Rh, double* RES,
                            int RESh, hipStream_t s, int mirror) {
  if (nch <= 0) return;
  hipLaunchKernelGGL(k_comm222ph_chunk, dim3(nch, B.ninst), dim3(256), 0, s, B, ch, fq, fql, fqi, items, W, Lh, Rh,
                     RES, RESh, mirror);
}

// ------------------------------------------------ 222_ph by block quadruples
// One wave (workgroup) per quadruple of blocks, or a part of it that fits its
// LDS; upper triangles of RES only.  The two W' sub-tiles of every
// (recoupling, J') slot are read along their own contiguous directions and
// meet in LDS (two additions onto zero: any order gives the same sum); then
// every output (J, i, j, k, l) sums its quadruple's values against the 6j
// coefficients of (J, slot).
// The chunk kernel above gathers single elements of W' (64 lanes, up to 64
// lines: the address path was busy 90 % of its time, 1.09 GB a launch at eMax 8
// for 0.41 GB of data); here the lanes run along rows of n_A n_C elements and
// neighbouring waves share what is left of a line (0.40 GB).  Bound now by
// vector instructions (index arithmetic: the vector units issue 60 % of the
// time with 16 waves a CU, on average over a launch, of the 29 that 5.6 KB of
// LDS each let in).  eMax 7 / 8 / 10: 69 / 182 / 1199 -> 46 / 93 / 642 us.  Tried: one
// workgroup per 3072 values of several quadruples, searched per lane (194 us at
// eMax 8, 3200 vector instructions a wave); a wave per quadruple in workgroups
// of four with 1024 values each (151 us: half the occupancy).
__device__ __forceinline__ float frcp(int n) { return __builtin_amdgcn_rcpf((float)n); }
__device__ __forceinline__ int fdiv(int x, float r) { return (int)(((float)x + 0.5f) * r); }   // x / n, r = frcp(n), x < 2^20
__device__ __forceinline__ void wave_lds_sync() {   // LDS of one wave is in order: hold the compiler only
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A W' sub-tile with the digits of its contiguous direction (f1 slow, f0
// fast, stride lf) and of the other one (s1, s0, ls): sizes, value-index
// strides, offsets of the members taken, the sign of its elements.  A tile of
// a row block before its column block is stored as it is (rows contiguous),
// else transposed with the factor -Lh Rh; of a block with itself the lower
// elements are read transposed.  All of it is wave-uniform.
struct PhbTile { int nf0, nf1, ns0, lf, ls, of, os, ef0, ef1, es0, es1; double sg; };
__device__ __forceinline__ PhbTile phb_tile(bool dir, int nr0, int nr1, int nc0, int nc1, int lr, int lc, int orow, int ocol,
                                            int er0, int er1, int ec0, int ec1, double mpm) {
  if (dir) return PhbTile{nr0, nr1, nc0, lr, lc, orow, ocol, er0, er1, ec0, ec1, 1.0};
  return PhbTile{nc0, nc1, nr0, lc, lr, ocol, orow, ec0, ec1, er0, er1, mpm};
}
// element e: its value index and its value; F, S the slot's first position in the two directions
__device__ __forceinline__ double phb_read(const PhbTile& T, float r0, float r1, float r2, int F, int S, unsigned wo,
                                           unsigned r, int e, const double* WCC, double mpm, int& ev) {
  const int q0 = fdiv(e, r0), f0 = e - q0 * T.nf0;
  const int q1 = fdiv(q0, r1), f1 = q0 - q1 * T.nf1;
  const int s1 = fdiv(q1, r2), s0 = q1 - s1 * T.ns0;
  ev = __mul24(f0, T.ef0) + __mul24(f1, T.ef1) + __mul24(s0, T.es0) + __mul24(s1, T.es1);
  const int x = F + __mul24(f1, T.lf) + f0, y = S + __mul24(s1, T.ls) + s0;
  const double w = WCC[wo + (unsigned)min(x, y) + __umul24((unsigned)max(x, y), r)];
  return (x <= y ? T.sg : mpm) * w;
}
// the slots [s0, s0 + n) of one recoupling: tiles T1, T2 added into v
__device__ __forceinline__ void phb_slots(const PhbTile& T1, const PhbTile& T2, bool d1, bool d2, const PhbSlot* ss, int s0,
                                          int n, int n4, const double* WCC, double mpm, int ph, double* v) {
  const float r4 = frcp(n4), a0 = frcp(T1.nf0), a1 = frcp(T1.nf1), a2 = frcp(T1.ns0);
  const float b0 = frcp(T2.nf0), b1 = frcp(T2.nf1), b2 = frcp(T2.ns0);
#pragma unroll 2
  for (int t = threadIdx.x; t < n * n4; t += 64) {
    const int q = fdiv(t, r4), e = t - q * n4, s = s0 + q;
    const PhbSlot S = ss[s];
    int v1, v2;
    const double w1 = phb_read(T1, a0, a1, a2, (d1 ? S.R1 : S.C1) + T1.of, (d1 ? S.C1 : S.R1) + T1.os, S.wo, S.r, e, WCC,
                               mpm, v1);
    const double w2 = phb_read(T2, b0, b1, b2, (d2 ? S.R2 : S.C2) + T2.of, (d2 ? S.C2 : S.R2) + T2.os, S.wo, S.r, e, WCC,
                               mpm, v2);
    unsafeAtomicAdd(&v[s * n4 + v1], w1);
    unsafeAtomicAdd(&v[s * n4 + v2], ph * w2);
  }
}

__global__ __launch_bounds__(64) void k_comm222ph_blk(DevBasis B, PhbPlan P, const double* WCC, int Lh, int Rh,
                                                      double* RES) {
  int inst;
  if (!batch_inst(B, inst)) return;
  WCC += (i64)inst * B.wclen;
  RES += (i64)inst * B.oplen;
  __shared__ double v[kPhbLds];
  __shared__ PhbSlot ss[kPhbSlots];
  __shared__ int mem[4 * kPhbMembers];   // members taken of the four blocks
  const int lane = threadIdx.x;
  const PhbQuad Q = P.quads[xcd_contig(blockIdx.x, gridDim.x)];   // neighbouring quadruples share lines of W' and RES
  const double mpm = -(double)(Lh * Rh);
  const int nA = Q.n & 255, nB = (Q.n >> 8) & 255, nC = (Q.n >> 16) & 255, nD = (Q.n >> 24) & 255;
  const int NA = Q.N & 255, NB = (Q.N >> 8) & 255, NC = (Q.N >> 16) & 255, ND = (Q.N >> 24) & 255;
  const int oA = Q.off & 255, oB = (Q.off >> 8) & 255, oC = (Q.off >> 16) & 255, oD = (Q.off >> 24) & 255;
  const int ji = Q.j & 255, jj = (Q.j >> 8) & 255, jk = (Q.j >> 16) & 255, jl = (Q.j >> 24) & 255;
  const int nin = Q.nin, ns = nin + Q.nout, n4 = nA * nB * nC * nD, nv = n4 * ns;
  const float r4 = frcp(n4);
  if (lane < ns) ss[lane] = P.slots[Q.slot0 + lane];
  {
    const int x = 8 * (lane >> 4), y = lane & 15;   // block, member
    if (y < (int)((Q.n >> x) & 255)) mem[lane] = P.mem[((Q.ob >> x) & 255) + ((Q.off >> x) & 255) + y];
  }
  for (int t = lane; t < nv; t += 64) v[t] = 0.0;
  wave_lds_sync();
  const int ph = m1pow((ji + jj + jk + jl) / 2);
  // value index of (i, j, k, l) at one slot: i + nA (k + nC (l + nD j));
  // in:  W'((k,i),(j,l)) and W'((l,j),(i,k));  out: W'((l,i),(j,k)) and W'((k,j),(i,l)).
  // Rows are ordered by blocks at every J', so one slot tells the order of all.
  const int eC = nA, eD = nA * nC, eB = nA * nC * nD;
  const float rA = frcp(nA), rC = frcp(nC), rD = frcp(nD);
  if (nin > 0) {
    const bool d1 = __builtin_amdgcn_readfirstlane(ss[0].R1 <= ss[0].C1), d2 = __builtin_amdgcn_readfirstlane(ss[0].R2 <= ss[0].C2);
    const PhbTile T1 = phb_tile(d1, nA, nC, nD, nB, NA, ND, oC * NA + oA, oB * ND + oD, 1, eC, eD, eB, mpm);
    const PhbTile T2 = phb_tile(d2, nB, nD, nC, nA, NB, NC, oD * NB + oB, oA * NC + oC, eB, eD, eC, 1, mpm);
    phb_slots(T1, T2, d1, d2, ss, 0, nin, n4, WCC, mpm, ph, v);
  }
  if (Q.nout > 0) {
    const bool d1 = __builtin_amdgcn_readfirstlane(ss[nin].R1 <= ss[nin].C1), d2 = __builtin_amdgcn_readfirstlane(ss[nin].R2 <= ss[nin].C2);
    const PhbTile T1 = phb_tile(d1, nA, nD, nC, nB, NA, NC, oD * NA + oA, oB * NC + oC, 1, eD, eC, eB, mpm);
    const PhbTile T2 = phb_tile(d2, nB, nC, nD, nA, NB, ND, oC * NB + oB, oA * ND + oD, eB, eC, eD, 1, mpm);
    phb_slots(T1, T2, d1, d2, ss, nin, Q.nout, n4, WCC, mpm, ph, v);
  }
  // 6j coefficients of (J, slot) behind the values
  double* cof = v + nv;
  const float rs = frcp(ns);
  for (int x = lane; x < ns * Q.nJ; x += 64) {
    const int jx = fdiv(x, rs), s = x - jx * ns, J = Q.lo + 2 * jx;
    cof[x] = s < nin ? -(double)m1pow((jl + jk + J) / 2) * sixj_tri(B, ji, jj, J, jl, jk, Q.jin + 2 * s)
                     : sixj_tri(B, ji, jj, J, jk, jl, Q.jout + 2 * (s - nin));
  }
  wave_lds_sync();
  for (int t = lane; t < n4 * Q.nJ; t += 64) {
    const int jx = fdiv(t, r4), e = t - jx * n4;
    const int J = Q.lo + 2 * jx;
    const int x1 = fdiv(e, rA), li = e - x1 * nA;
    const int x2 = fdiv(x1, rC), lk = x1 - x2 * nC;
    const int lj = fdiv(x2, rD), ll = x2 - lj * nD;
    int i = mem[li], j = mem[kPhbMembers + lj], k = mem[2 * kPhbMembers + lk], l = mem[3 * kPhbMembers + ll];
    const int cp = (i >> 8) + (j >> 8), cq = (k >> 8) + (l >> 8);
    i &= 255; j &= 255; k &= 255; l &= 255;
    // pairs of one block are taken in orbit order once, and of {A, B} ==
    // {C, D} the upper triangle
    if (((Q.same & 1) && i > j) || ((Q.same & 2) && k > l)) continue;
    const int ip = B.xmap[(i * B.N + j) * B.nJ + (J >> 1)];
    const int iq = B.xmap[(k * B.N + l) * B.nJ + (J >> 1)];
    const bool up = cp < cq || (cp == cq && ip <= iq);   // stored as (ij, kl)
    if ((Q.same & 4) && !up) continue;
    const double* cf = cof + jx * ns;
    const double* vp = v + e;
    double sm = 0.0;
    for (int s = 0; s < ns; ++s) sm = fma(cf[s], vp[s * n4], sm);
    if (i == j) sm *= IMSRG_INV_SQRT2_REF;
    if (k == l) sm *= IMSRG_INV_SQRT2_REF;
    // <ij| = -(-1)^((ji + jj - J) / 2) <ji|, and for kl; the lower element by
    // RES(kl, ij) = -Lh Rh RES(ij, kl)
    int neg = 0;
    if (i > j) neg ^= 1 + (ji + jj - J) / 2;
    if (k > l) neg ^= 1 + (jk + jl - J) / 2;
    if (neg & 1) sm = -sm;
    if (!up) sm *= mpm;
    const int qc = 3 * J + Q.m;
    const int clo = up ? cp : cq, chi = up ? cq : cp;
    const int row = up ? ip : iq, col = up ? iq : ip;
    double* X = RES + B.goff[qc * 6 + blk_of(clo, chi)] + row + (i64)col * B.dims[qc * 3 + clo];
    *X = *X + sm;
  }
}

void launch_comm222ph_blk(const DevBasis& B, const PhbPlan& P, const double* W, int Lh, int Rh, double* RES,
                          hipStream_t s) {
  if (P.nquads <= 0) return;
  hipLaunchKernelGGL(k_comm222ph_blk, dim3(P.nquads, B.ninst), dim3(64), 0, s, B, P, W, Lh, Rh, RES);
}

// lower triangle of every square block (pppp, phph, hhhh) from its upper
// triangle: X(y, x) = herm X(x, y) for x < y, by 64 x 64 tile pairs (tile
// rows ti <= tile columns tj; task.pad = block g) through LDS, coalesced
// both ways.  Lets the fused commutator's 122 and 222_ph write only the
// upper triangles.
__global__ __launch_bounds__(256) void k_sym_lower(DevBasis B, const PairTask* tasks, double* RES, int herm) {
  __shared__ double T[64][65];
  int inst;
  if (!batch_inst(B, inst)) return;
  RES += (i64)inst * B.oplen;
  const PairTask t = tasks[blockIdx.x];
  const int q = t.q, g = t.pad;
  const int n = brows(B, q, g);
  double* X = RES + B.goff[q * 6 + g];
  const int x0 = t.ti * 64, y0 = t.tj * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int c = ty; c < 64; c += 4) {   // upper tile, column y0 + c
    const int x = x0 + tx, y = y0 + c;
    T[c][tx] = (x < n && y < n && x < y) ? X[x + (i64)y * n] : 0.0;
  }
  __syncthreads();
  for (int c = ty; c < 64; c += 4) {   // lower tile, column x0 + c
    const int yy = y0 + tx, xx = x0 + c;
    if (yy < n && xx < n && xx < yy) X[yy + (i64)xx * n] = herm * T[tx][c];
  }
}

void launch_sym_lower(const DevBasis& B, const PairTask* t, int nt, double* RES, int herm, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_sym_lower, dim3(nt, B.ninst), dim3(256), 0, s, B, t, RES, herm);
}

// =========================================================== Pandya forward
// calculate_cross_coupled, cross_coupled.f90:1190-1300.  One thread per
// CCX(q1)(r, nb) element; r = ordered pair (a,b), nb = (p,h).
__device__ __forceinline__ void d_pandya(DevBasis B, const CCTask* tasks, const double* op, int herm, double* CC,
                                         int bx, int nbx) {
  int inst;
  if (!batch_inst(B, inst)) return;
  op += (i64)inst * B.oplen;
  CC += (i64)inst * B.cclen;
  const CCTask t = tasks[xcd_contig(bx, nbx)];
  const int q1 = t.q1;
  const int r = B.rlen[q1], nc = B.ncol[q1];
  const i64 e = (i64)t.start + threadIdx.x;
  if (e >= (i64)r * nc) return;
  const int R = (int)(e % r), NB = (int)(e / r);
  int a, b, p, h;
  unpack(B.ccrows[B.ccrowoff[q1] + R], a, b);
  unpack(B.cccols[B.cccoloff[q1] + NB], p, h);
  const int JC = B.ccJ[q1];
  const int ja = B.jj[a], jb = B.jj[b], jp = B.jj[p], jh = B.jj[h];
  const int la = B.ll[a], lb = B.ll[b], lp = B.ll[p], lh = B.ll[h];
  const int ta = B.tz[a], tb = B.tz[b], tp = B.tz[p], th = B.tz[h];
  double val = 0.0;
  if ((((la + lh) & 1) == ((lb + lp) & 1)) && (ta + th == tb + tp)) {
    const int Jmin = max(abs(jp - jb), abs(ja - jh));
    const int Jmax = min(jp + jb, ja + jh);
    double sm = 0.0;
    for (int JT = Jmin; JT <= Jmax; JT += 2)
      sm = sm + (double)(m1pow(JT / 2) * (JT + 1)) * sixj(B, jp, jh, JC, ja, jb, JT) *
                    v_elem(B, op, herm, h, a, p, b, JT);
    val = sm * m1pow((jh + jb + JC) / 2) * 1.0 * sqrt(JC + 1.0);
  }
  CC[B.ccoff[q1] + R + (i64)NB * r] = val;
}

__global__ __launch_bounds__(256) void k_pandya(DevBasis B, const CCTask* tasks, const double* op, int herm,
                                                double* CC) {
  d_pandya(B, tasks, op, herm, CC, blockIdx.x, gridDim.x);
}

void launch_pandya(const DevBasis& B, const CCTask* t, int nt, const double* op, int herm, double* CC,
                   hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_pandya, dim3(nt, B.ninst), dim3(kTile), 0, s, B, t, op, herm, CC);
}

// ============================================================ commutator_111
// commutators.f90:36-80.  One wave per one-body output (assigns); the lanes
// split the intermediate orbit k and the partial dot products are reduced
// across the wave.
__device__ __forceinline__ void d_comm111(DevBasis B, const double* L, int Lh, const double* R, int Rh,
                                          double* RES, int bx) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  RES += (i64)inst * B.oplen;
  const int A = B.A, P = B.P;
  const i64 idx = (i64)bx * 4 + (threadIdx.x >> 6);   // wave-uniform
  const int lane = threadIdx.x & 63;
  const double *Lhh = L + B.off_fhh, *Lph = L + B.off_fph, *Lpp = L + B.off_fpp;
  const double *Rhh = R + B.off_fhh, *Rph = R + B.off_fph, *Rpp = R + B.off_fpp;
  double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
  if (idx < (i64)A * A) {
    const int i = (int)(idx % A), j = (int)(idx / A);
    for (int k = lane; k < A; k += 64) {
      s0 += Lhh[i + k * A] * Rhh[k + j * A];
      s1 += Lhh[j + k * A] * Rhh[k + i * A];
    }
    for (int k = lane; k < P; k += 64) {
      s2 += Lph[k + (i64)i * P] * Rph[k + (i64)j * P];
      s3 += Lph[k + (i64)j * P] * Rph[k + (i64)i * P];
    }
    s0 = wave_sum(s0); s1 = wave_sum(s1); s2 = wave_sum(s2); s3 = wave_sum(s3);
    if (lane == 0) RES[B.off_fhh + idx] = s0 + s2 * Lh - (s1 * Lh + s3) * Rh;
    return;
  }
  if (idx < (i64)A * A + (i64)P * A) {
    const i64 x = idx - (i64)A * A;
    const int a = (int)(x % P), i = (int)(x / P);
    for (int k = lane; k < A; k += 64) {
      s0 += Lph[a + (i64)k * P] * Rhh[k + i * A];
      s1 += Rph[a + (i64)k * P] * Lhh[k + i * A];
    }
    for (int k = lane; k < P; k += 64) {
      s2 += Lpp[a + (i64)k * P] * Rph[k + (i64)i * P];
      s3 += Rpp[a + (i64)k * P] * Lph[k + (i64)i * P];
    }
    s0 = wave_sum(s0); s1 = wave_sum(s1); s2 = wave_sum(s2); s3 = wave_sum(s3);
    if (lane == 0) RES[B.off_fph + x] = (s0 + s2) - s1 - s3;
    return;
  }
  if (idx < (i64)A * A + (i64)P * A + (i64)P * P) {
    const i64 x = idx - (i64)A * A - (i64)P * A;
    const int a = (int)(x % P), b = (int)(x / P);
    for (int k = lane; k < A; k += 64) {
      s0 += Lph[a + (i64)k * P] * Rph[b + (i64)k * P];
      s1 += Lph[b + (i64)k * P] * Rph[a + (i64)k * P];
    }
    for (int k = lane; k < P; k += 64) {
      s2 += Lpp[a + (i64)k * P] * Rpp[k + (i64)b * P];
      s3 += Lpp[b + (i64)k * P] * Rpp[k + (i64)a * P];
    }
    s0 = wave_sum(s0); s1 = wave_sum(s1); s2 = wave_sum(s2); s3 = wave_sum(s3);
    if (lane == 0) RES[B.off_fpp + x] = s0 * Rh + s2 - (s1 + s3 * Rh) * Lh;
  }
}

__global__ __launch_bounds__(256) void k_comm111(DevBasis B, const double* L, int Lh, const double* R, int Rh,
                                                 double* RES) {
  d_comm111(B, L, Lh, R, Rh, RES, blockIdx.x);
}

void launch_comm111(const DevBasis& B, const double* L, int Lh, const double* R, int Rh, double* RES,
                    hipStream_t s) {
  const i64 n = (i64)B.A * B.A + (i64)B.P * B.A + (i64)B.P * B.P;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_comm111, dim3((unsigned)((n + 3) / 4), B.ninst), dim3(256), 0, s, B, L, Lh, R, Rh, RES);
}

__device__ double block_sum(double v, double* red);

// one-body result of 121 / 221: RES(p,q) += add and the herm-symmetric fill
__device__ __forceinline__ void onebody_update(const DevBasis& B, const OneTask& t, double add, double* RES,
                                               int RESh) {
  if (t.kind == 0) {
    double* F = RES + B.off_fhh;
    const i64 o = t.pi + (i64)t.qi * B.A;
    F[o] = F[o] + add;
    F[t.qi + (i64)t.pi * B.A] = F[o] * RESh;
  } else if (t.kind == 1) {
    double* F = RES + B.off_fpp;
    const i64 o = t.pi + (i64)t.qi * B.P;
    F[o] = F[o] + add;
    F[t.qi + (i64)t.pi * B.P] = F[o] * RESh;
  } else {
    double* F = RES + B.off_fph;
    const i64 o = t.pi + (i64)t.qi * B.P;
    F[o] = F[o] + add;
  }
}

// ============================================================ commutator_121
// commutators.f90:83-280 (accumulates).  One workgroup per one-body output
// (p, q); its threads take the (particle a, hole i, J) terms, with (a, i)
// from the list of particle-hole pairs inside one (l, j, tz) block (the
// only pairs the reference's loop keeps), tree-reduced in LDS.
// Its terms go round kOneLanes lanes; a workgroup has that many threads or half
// of them with two lanes each (onebody_threads), and the sums are the same.
constexpr int kOneLanes = 512;
__device__ __forceinline__ void d_comm121(DevBasis B, const OneTask* tasks, const double* L, int Lh,
                                          const double* R, int Rh, double* RES, int RESh, int bx, double* red) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  RES += (i64)inst * B.oplen;
  const OneTask t = tasks[bx];
  const int pk = t.pk, qk = t.qk, jq = B.jj[qk];
  const double* Lph = L + B.off_fph;
  const double* Rph = R + B.off_fph;
  const int JS = B.jsmax;
  double sum = 0.0;
  for (int ln = threadIdx.x; ln < kOneLanes; ln += blockDim.x) {
    double v = 0.0;
    for (int x = ln; x < B.nphp * JS; x += kOneLanes) {
      const int pr = x / JS, js = x % JS;
      const int a = B.php[2 * pr], i = B.php[2 * pr + 1];
      const int ak = B.parts[a], ik = B.holes[i];
      const int ji = B.jj[ik];
      const int JT = abs(ji - jq) + 2 * js;
      if (JT > ji + jq) continue;
      const VPos p1 = vpos(B, ak, pk, ik, qk, JT);
      const VPos p2 = vpos(B, ik, pk, ak, qk, JT);
      const double la = Lph[a + (i64)i * B.P], ra = Rph[a + (i64)i * B.P];
      v = v + (JT + 1) * (la * (Lh * vat(p1, R, Rh) - vat(p2, R, Rh)) - ra * (Rh * vat(p1, L, Lh) - vat(p2, L, Lh)));
    }
    sum += v;
  }
  const double sm = block_sum(sum, red);
  if (threadIdx.x == 0) onebody_update(B, t, sm / (B.jj[pk] + 1.0), RES, RESh);
}

// Threads of a workgroup of 121 and 221, n terms a result.  A thread's terms run
// one after the other, each a chain of dependent reads, so one lane a thread is
// faster while the launch is one round of workgroups (four of 512 threads a CU,
// 1024 in all) and there are terms for the second half; beyond, idle threads
// hold the place of the next results.  256 / 512 threads, us, 121 and 221: eMax 8 16O
// (190 results) 9.4 / 7.1 and 30.1 / 20.6, four instances 13.3 / 10.9 and 48.6 / 33.6,
// eight 16.4 / 22.6 and 58.2 / 68.7; eMax 10 (322) 13.1 / 10.3 and 46.1 / 30.0, four
// 21.9 / 30.3 and 81.3 / 83.5; eMax 6 (100; 121 has 196 terms) 64 instances 40.6 / 71.2
// and 119 / 150, eight 9.0 / 14.2 and 27.0 / 24.3.
static int onebody_threads(const DevBasis& B, int nt, int n) {
  return n > kOneLanes / 2 && (i64)nt * B.ninst <= 1024 ? kOneLanes : kOneLanes / 2;
}

__global__ __launch_bounds__(512) void k_comm121(DevBasis B, const OneTask* tasks, const double* L, int Lh,
                                                 const double* R, int Rh, double* RES, int RESh) {
  __shared__ double red[kOneLanes];
  d_comm121(B, tasks, L, Lh, R, Rh, RES, RESh, blockIdx.x, red);
}

void launch_comm121(const DevBasis& B, const OneTask* t, int nt, const double* L, int Lh, const double* R,
                    int Rh, double* RES, int RESh, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_comm121, dim3(nt, B.ninst), dim3(onebody_threads(B, nt, B.nphp * B.jsmax)), 0, s, B, t, L, Lh, R, Rh, RES, RESh);
}

// ============================================================ commutator_221
// commutators.f90:435-578 (accumulates; reads w1/w2 of 222_pp_hh, herm 1).
// One workgroup per one-body output; its threads take the (intermediate
// orbit c, 2J) terms (holes c with w1, particles c with w2), tree-reduced.
// Elements of w2's pppp blocks (W2 = Rh L3 R3^T, rank nh) are formed from L
// and R here, so 222_pp_hh need not store that block.
__device__ __forceinline__ double w2_elem(const DevBasis& B, const double* w2, const double* L, const double* R,
                                          int Rh, int a, int b, int c, int d, int J) {
  const VPos p = vpos(B, a, b, c, d, J);
  if (p.off < 0) return 0.0;
  const int C1 = B.con[a] + B.con[b], C2 = B.con[c] + B.con[d];
  if (C1 != 0 || C2 != 0) return vat(p, w2, 1);
  const int q = 3 * J + 2 * ((B.tz[a] + B.tz[b]) / 2 + 1) + ((B.ll[a] + B.ll[b]) & 1);
  const int np = B.dims[q * 3], nh = B.dims[q * 3 + 2];
  const i64 o3 = B.goff[q * 6 + 2];
  const i64 rel = p.off - B.goff[q * 6 + 0];
  const int x = (int)(rel % np), y = (int)(rel / np);
  double s = 0.0;
  for (int h = 0; h < nh; ++h) s += L[o3 + x + (i64)h * np] * R[o3 + y + (i64)h * np];
  return (s * Rh) * p.pre;
}

__device__ __forceinline__ void d_comm221(DevBasis B, const OneTask* tasks, const double* L, int Lh,
                                          const double* R, int Rh, const double* w1, const double* w2,
                                          double* RES, int RESh, int bx, double* red) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  w1 += (i64)inst * B.oplen;
  w2 += (i64)inst * B.oplen;
  RES += (i64)inst * B.oplen;
  const OneTask t = tasks[bx];
  const int ik = t.pk, jk = t.qk, ji = B.jj[ik];
  const int pm = Lh * Rh;
  const bool both = (t.kind != 2);
  const int JS = B.jsmax;
  double sum = 0.0;
  // item (c, J): intermediate orbit c (holes first, with w1; then particles,
  // with w2) and one 2J of its coupling to i
  for (int ln = threadIdx.x; ln < kOneLanes; ln += blockDim.x) {
    double v = 0.0;
    for (int y = ln; y < B.N * JS; y += kOneLanes) {
      const int x = y / JS;
      const bool hole = x < B.A;
      const int ck = hole ? B.holes[x] : B.parts[x - B.A];
      const int jc = B.jj[ck];
      const int JT = abs(jc - ji) + 2 * (y % JS);
      if (JT > jc + ji) continue;
      if (hole) {
        if (both)
          v = v + (v_elem(B, w1, 1, ck, ik, ck, jk, JT) - pm * v_elem(B, w1, 1, ck, jk, ck, ik, JT)) * (JT + 1);
        else
          v = v + v_elem(B, w1, 1, ck, ik, ck, jk, JT) * (JT + 1);
      } else {
        if (both)
          v = v + (w2_elem(B, w2, L, R, Rh, ck, ik, ck, jk, JT) - pm * w2_elem(B, w2, L, R, Rh, ck, jk, ck, ik, JT)) *
                      (JT + 1);
        else
          v = v + w2_elem(B, w2, L, R, Rh, ck, ik, ck, jk, JT) * (JT + 1);
      }
    }
    sum += v;
  }
  const double sm = block_sum(sum, red);
  if (threadIdx.x == 0) onebody_update(B, t, sm / (ji + 1.0), RES, RESh);
}

__global__ __launch_bounds__(512) void k_comm221(DevBasis B, const OneTask* tasks, const double* L, int Lh,
                                                 const double* R, int Rh, const double* w1, const double* w2,
                                                 double* RES, int RESh) {
  __shared__ double red[kOneLanes];
  d_comm221(B, tasks, L, Lh, R, Rh, w1, w2, RES, RESh, blockIdx.x, red);
}

void launch_comm221(const DevBasis& B, const OneTask* t, int nt, const double* L, int Lh, const double* R, int Rh,
                    const double* w1, const double* w2, double* RES, int RESh, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_comm221, dim3(nt, B.ninst), dim3(onebody_threads(B, nt, B.N * B.jsmax)), 0, s, B, t, L, Lh, R, Rh, w1, w2, RES, RESh);
}

// ================================================= commutator_110 + 220 (E0)
// commutators.f90:10-33 and 399-432.  Workgroup q < nblocks: channel q's
// 220 sum times (2J+1); workgroup nblocks: the 110 sum.
__device__ double block_sum(double v, double* red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

__device__ __forceinline__ void d_e0_partials(DevBasis B, const double* L, int Lh, const double* R, int Rh,
                                              double* part, int bx, double* red) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  part += (i64)inst * B.spart;
  const int q = bx;
  double v = 0.0;
  if (q < B.nblocks) {
    const int np = B.dims[q * 3], nh = B.dims[q * 3 + 2];
    const double* L3 = L + B.goff[q * 6 + 2];
    const double* R3 = R + B.goff[q * 6 + 2];
    for (i64 x = threadIdx.x; x < (i64)np * nh; x += blockDim.x) v = v - L3[x] * R3[x] * Rh;
    const double s = block_sum(v, red);
    if (threadIdx.x == 0) part[q] = s * (B.chJ[q] + 1);
  } else {
    const double* Lph = L + B.off_fph;
    const double* Rph = R + B.off_fph;
    for (i64 x = threadIdx.x; x < (i64)B.P * B.A; x += blockDim.x) {
      const int hk = B.holes[(int)(x / B.P)];
      v = v + (Lph[x] * Rph[x] * Lh - Rph[x] * Lph[x] * Rh) * (B.jj[hk] + 1);
    }
    const double s = block_sum(v, red);
    if (threadIdx.x == 0) part[B.nblocks] = s;
  }
}

__global__ __launch_bounds__(256) void k_e0_partials(DevBasis B, const double* L, int Lh, const double* R,
                                                     int Rh, double* part) {
  __shared__ double red[256];
  d_e0_partials(B, L, Lh, R, Rh, part, blockIdx.x, red);
}

// dst = [use110] part[n] + [use220] 2 * sum(part[0..n-1])   (one workgroup)
__device__ __forceinline__ void d_e0_final(const double* part, int n, int use220, int use110, double* dst,
                                           int accumulate, i64 spart, i64 sdst, const int* act, double* red) {
  int inst;
  if (!batch_on(act, inst)) return;
  part += (i64)inst * spart;
  dst += (i64)inst * sdst;
  double v = 0.0;
  for (int x = threadIdx.x; x < n; x += blockDim.x) v += part[x];
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) {
    const double e110 = use110 ? part[n] : 0.0;
    const double e220 = use220 ? s * 2.0 : 0.0;
    const double e = e110 + e220;
    dst[0] = accumulate ? dst[0] + e : e;
  }
}

__global__ __launch_bounds__(256) void k_e0_final(const double* part, int n, int use220, int use110, double* dst,
                                                  int accumulate, i64 spart, i64 sdst, const int* act) {
  __shared__ double red[256];
  d_e0_final(part, n, use220, use110, dst, accumulate, spart, sdst, act, red);
}

void launch_e0_partials(const DevBasis& B, const double* L, int Lh, const double* R, int Rh, double* part,
                        hipStream_t s) {
  hipLaunchKernelGGL(k_e0_partials, dim3(B.nblocks + 1, B.ninst), dim3(256), 0, s, B, L, Lh, R, Rh, part);
}

void launch_e0_final(const double* part, int nblocks, int use220, int use110, double* dst, int accumulate,
                     hipStream_t s) {
  hipLaunchKernelGGL(k_e0_final, dim3(1), dim3(256), 0, s, part, nblocks, use220, use110, dst, accumulate, (i64)0,
                     (i64)0, (const int*)nullptr);
}
void launch_e0_final_b(const DevBasis& B, const double* part, int use220, int use110, double* dst, int accumulate,
                       hipStream_t s) {
  hipLaunchKernelGGL(k_e0_final, dim3(1, B.ninst), dim3(256), 0, s, part, B.nblocks, use220, use110, dst, accumulate,
                     B.spart, B.oplen, B.act);
}

// ======================================== 222_pp_hh pppp block epilogue
// commutators.f90:611-668.  The grouped GEMM leaves C = W1 - W2 =
// L1 R1 - Rh L3 R3^T in w1's pppp block; RES1 += C - pm C^T.  Tile pair
// (I,J), I <= J, of 64 x 64: both C tiles are staged through LDS so every
// global access is a contiguous column run.  The reference's W1 and W2 are
// left in w1 / w2 (W2 formed here, rank nh).
// Bound by latency at small sizes: a thread of one of two halves (tile (I, J)
// and tile (J, I)) issues the 16 loads of its elements and of RES at once, and
// W2's columns of R3 are uniform to a wave (one row of L3 a lane).  With a
// load, a test and a W2 sum per element, one after the other, 222_pp_hh took
// 315 us at eMax 8, now 261.
__global__ __launch_bounds__(512) void k_pppp_sym(DevBasis B, const PairTask* tasks, const double* L, int Lh,
                                                  const double* R, int Rh, double* RES, double* w1, double* w2) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  RES += (i64)inst * B.oplen;
  w1 += (i64)inst * B.oplen;
  w2 += (i64)inst * B.oplen;
  __shared__ double S[2][64][65];   // S[half][x][y] = C(X0 + x, Y0 + y) of the half's tile
  const PairTask t = tasks[blockIdx.x];
  const int q = t.q;
  const int np = B.dims[q * 3], nh = B.dims[q * 3 + 2];
  const i64 o1 = B.goff[q * 6 + 0], o3 = B.goff[q * 6 + 2];
  const double *L3 = L + o3, *R3 = R + o3;
  double* Cm = w1 + o1;
  double* X1 = RES + o1;
  double* W21 = w2 + o1;
  const int pm = Lh * Rh;
  const bool diag = t.ti == t.tj;
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int x = threadIdx.x & 63, y0 = 16 * (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3);
  const int X0 = (half ? t.tj : t.ti) * 64, Y0 = (half ? t.ti : t.tj) * 64;
  const int gx = X0 + x, cx = min(gx, np - 1);
  double c[16], u[16];
  if (!(diag && half)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const i64 o = cx + (i64)min(Y0 + y0 + r, np - 1) * np;
      c[r] = Cm[o];
      u[r] = X1[o];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) S[half][x][y0 + r] = c[r];
  }
  __syncthreads();
  if (diag && half) return;
  double w[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) w[r] = 0.0;
  for (int h = 0; h < nh; ++h) {
    const double l = L3[cx + (i64)h * np];
#pragma unroll
    for (int r = 0; r < 16; ++r) w[r] += l * R3[min(Y0 + y0 + r, np - 1) + (i64)h * np];
  }
  const double (*St)[65] = S[diag ? 0 : 1 - half];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int gy = Y0 + y0 + r;
    if (gx < np && gy < np) {
      const i64 o = gx + (i64)gy * np;
      const double w2v = w[r] * Rh;
      X1[o] = u[r] + c[r] - St[y0 + r][x] * pm;
      Cm[o] = c[r] + w2v;
      W21[o] = w2v;
    }
  }
}

// The same epilogue when w1 is not rewritten (the flow's commutator): one
// workgroup per output tile (two per off-diagonal pair, blockIdx.x = 2 task
// + side), its own C tile read straight from memory and only the tile whose
// transpose it needs staged in LDS (33 KB instead of 66 KB: twice the
// workgroups per CU).  Same arithmetic as k_pppp_sym.  A load and a test
// at a time it took 14.2 us (eMax 6), 30.7 (8), 125 (10); now 6.4, 22.4, 112.
__device__ __forceinline__ void d_pppp_sym1(DevBasis B, const PairTask* tasks, double* RES, const double* w1,
                                            int pm, int upper_only, int bx, double (*S)[65]) {
  int inst;
  if (!batch_inst(B, inst)) return;
  RES += (i64)inst * B.oplen;
  w1 += (i64)inst * B.oplen;
  // S[x][y] = C(A0 + x, B0 + y), the transposed source tile
  // upper_only: one workgroup per tile pair for its upper tile (the caller
  // fills the lower triangles afterwards), else two, the second for the
  // lower tile
  const PairTask t = tasks[upper_only ? bx : bx >> 1];
  const int side = upper_only ? 0 : (bx & 1);
  if (side == 1 && t.ti == t.tj) return;
  const int q = t.q;
  const int np = B.dims[q * 3];
  const i64 o1 = B.goff[q * 6 + 0];
  const double* Cm = w1 + o1;
  double* X1 = RES + o1;
  // output tile rows R0.., cols C0..; source tile rows C0.., cols R0..
  const int R0 = (side == 0 ? t.ti : t.tj) * 64, C0 = (side == 0 ? t.tj : t.ti) * 64;
  // every load of a thread before the barrier, at valid addresses
  const int x = threadIdx.x & 63, y0 = threadIdx.x >> 6;
  double c[16], u[16], v[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int y = y0 + 4 * r;
    const i64 o = min(R0 + x, np - 1) + (i64)min(C0 + y, np - 1) * np;
    v[r] = Cm[min(C0 + x, np - 1) + (i64)min(R0 + y, np - 1) * np];
    c[r] = Cm[o];
    u[r] = X1[o];
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) S[x][y0 + 4 * r] = v[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int y = y0 + 4 * r, gx = R0 + x, gy = C0 + y;
    if (gx < np && gy < np) X1[gx + (i64)gy * np] = u[r] + c[r] - S[y][x] * pm;
  }
}

__global__ __launch_bounds__(256) void k_pppp_sym1(DevBasis B, const PairTask* tasks, double* RES,
                                                   const double* w1, int pm, int upper_only) {
  __shared__ double S[64][65];
  d_pppp_sym1(B, tasks, RES, w1, pm, upper_only, blockIdx.x, S);
}

void launch_pppp_sym(const DevBasis& B, const PairTask* t, int nt, const double* L, int Lh, const double* R, int Rh,
                     double* RES, double* w1, double* w2, int ref_outputs, hipStream_t s) {
  if (nt <= 0) return;
  if (ref_outputs != 1) {
    const int upper_only = ref_outputs == 2 ? 1 : 0;
    hipLaunchKernelGGL(k_pppp_sym1, dim3(upper_only ? nt : 2 * nt, B.ninst), dim3(256), 0, s, B, t, RES,
                       (const double*)w1, Lh * Rh, upper_only);
    return;
  }
  hipLaunchKernelGGL(k_pppp_sym, dim3(nt, B.ninst), dim3(512), 0, s, B, t, L, Lh, R, Rh, RES, w1, w2);
}

// ================================ 222_pp_hh epilogue of the small blocks
// commutators.f90:636-764 after the grouped GEMMs:
//   g == 1: region gam2|gam3 (np x (nb+nh)); w1 already holds
//           L1 [R2|R3] - R1 [L2|L3]; adds the rank-nh parts W2 and RES.
//   g == 3 / 4 / 5: gam4 / gam5 / gam6 from P = [L2|L3]^T [R2|R3].
// P = [L2|L3]^T [R2|R3] (nbh x nbh) element (x, y): sum of the split-K slabs
__device__ __forceinline__ double pval(const double* Pq, int nbh, int ks, int x, int y) {
  double v = 0.0;
  for (int s = 0; s < ks; ++s) v += Pq[(i64)s * nbh * nbh + x + (i64)y * nbh];
  return v;
}

__device__ __forceinline__ void d_pphh_epilogue(DevBasis B, const SegTask* tasks, const double* L, int Lh,
                                                const double* R, int Rh, double* RES, double* w1, double* w2,
                                                const double* Pscr, const i64* poff, const int* k3ks,
                                                const double* K2scr, const i64* k2off, const int* k2ks, int bx) {
  int inst;
  if (!batch_inst(B, inst)) return;
  L += (i64)inst * B.oplen;
  R += (i64)inst * B.oplen;
  RES += (i64)inst * B.oplen;
  w1 += (i64)inst * B.oplen;
  w2 += (i64)inst * B.oplen;
  Pscr += (i64)inst * B.spscr;
  K2scr += (i64)inst * B.sk2scr;
  const SegTask t = tasks[bx];
  const i64 e = (i64)t.start + threadIdx.x;
  if (e >= t.cnt) return;
  const int q = t.q;
  const int np = B.dims[q * 3], nb = B.dims[q * 3 + 1], nh = B.dims[q * 3 + 2];
  const int pm = Lh * Rh;
  const i64* go = B.goff + q * 6;
  const double *L3 = L + go[2], *R3 = R + go[2], *L5 = L + go[4], *R5 = R + go[4], *L6 = L + go[5],
               *R6 = R + go[5];
  if (t.g == 1) {
    const int x = (int)(e % np), y = (int)(e / np);
    double w2v;
    if (y < nb) {
      double s1 = 0.0, s2 = 0.0;
      for (int h = 0; h < nh; ++h) {
        s1 += L3[x + (i64)h * np] * R6[y + (i64)h * nb];
        s2 += R3[x + (i64)h * np] * L6[y + (i64)h * nb];
      }
      w2v = Rh * s1 + (-1.0 * Lh) * s2;
    } else {
      const int hp = y - nb;
      double s1 = 0.0, s2 = 0.0;
      for (int h = 0; h < nh; ++h) {
        s1 += L3[x + (i64)h * np] * R5[h + (i64)hp * nh];
        s2 += R3[x + (i64)h * np] * L5[h + (i64)hp * nh];
      }
      w2v = s1 + (-1.0) * s2;
    }
    // W1 = L1 [R2|R3] - R1 [L2|L3]: sum of the split-K slabs
    double w1v = 0.0;
    const double* K2q = K2scr + k2off[q];
    const i64 slab = (i64)np * (nb + nh);
    for (int s = 0; s < k2ks[q]; ++s) w1v += K2q[s * slab + e];
    const i64 o = go[1] + e;
    RES[o] = RES[o] + w1v - w2v;
    w1[o] = w1v;
    w2[o] = w2v;
    return;
  }
  const int nbh = nb + nh;
  const double* Pq = Pscr + poff[q];
  const int ks = k3ks[q];
  if (t.g == 3) {   // gam4, nb x nb
    const int x = (int)(e % nb), y = (int)(e / nb);
    double sxy = 0.0, syx = 0.0;
    for (int h = 0; h < nh; ++h) {
      sxy += L6[x + (i64)h * nb] * R6[y + (i64)h * nb];
      syx += L6[y + (i64)h * nb] * R6[x + (i64)h * nb];
    }
    const double w1xy = pval(Pq, nbh, ks, x, y) * Lh, w1yx = pval(Pq, nbh, ks, y, x) * Lh;
    const double w2xy = sxy * Rh, w2yx = syx * Rh;
    const i64 o = go[3] + e;
    RES[o] = RES[o] + w1xy - w2xy - (w1yx - w2yx) * pm;
    w1[o] = w1xy;
    w2[o] = w2xy;
    return;
  }
  if (t.g == 4) {   // gam5, nh x nh
    const int a = (int)(e % nh), b = (int)(e / nh);
    double sab = 0.0, sba = 0.0;
    for (int h = 0; h < nh; ++h) {
      sab += L5[a + (i64)h * nh] * R5[h + (i64)b * nh];
      sba += L5[b + (i64)h * nh] * R5[h + (i64)a * nh];
    }
    const double w1ab = pval(Pq, nbh, ks, nb + a, nb + b) * Lh, w1ba = pval(Pq, nbh, ks, nb + b, nb + a) * Lh;
    const i64 o = go[4] + e;
    RES[o] = RES[o] + w1ab - sab - (w1ba - sba) * pm;
    w1[o] = w1ab;
    w2[o] = sab;
    return;
  }
  {   // gam6, nb x nh
    const int x = (int)(e % nb), h = (int)(e / nb);
    double s1 = 0.0, s2 = 0.0;
    for (int hp = 0; hp < nh; ++hp) {
      s1 += L6[x + (i64)hp * nb] * R5[hp + (i64)h * nh];
      s2 += R6[x + (i64)hp * nb] * L5[hp + (i64)h * nh];
    }
    const double w1v = Lh * pval(Pq, nbh, ks, x, nb + h) + (-1.0 * Rh) * pval(Pq, nbh, ks, nb + h, x);
    const double w2v = s1 + (-1.0) * s2;
    const i64 o = go[5] + e;
    RES[o] = RES[o] + w1v - w2v;
    w1[o] = w1v;
    w2[o] = w2v;
  }
}

__global__ __launch_bounds__(256) void k_pphh_epilogue(DevBasis B, const SegTask* tasks, const double* L, int Lh,
                                                       const double* R, int Rh, double* RES, double* w1,
                                                       double* w2, const double* Pscr, const i64* poff,
                                                       const int* k3ks, const double* K2scr, const i64* k2off,
                                                       const int* k2ks) {
  d_pphh_epilogue(B, tasks, L, Lh, R, Rh, RES, w1, w2, Pscr, poff, k3ks, K2scr, k2off, k2ks, blockIdx.x);
}

void launch_pphh_epilogue(const DevBasis& B, const SegTask* t, int nt, const double* L, int Lh, const double* R,
                          int Rh, double* RES, double* w1, double* w2, const double* Pscr, const i64* poff,
                          const int* k3ks, const double* K2scr, const i64* k2off, const int* k2ks, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_pphh_epilogue, dim3(nt, B.ninst), dim3(256), 0, s, B, t, L, Lh, R, Rh, RES, w1, w2, Pscr, poff, k3ks,
                     K2scr, k2off, k2ks);
}

// ================================================ streaming algebra / norm
// add_sq_op, basic_IMSRG.f90:3551-3583:  C = A*ax + B*bx
__global__ __launch_bounds__(256) void k_axpy(i64 n, const double* A, double ax, const double* Bv, double bx,
                                              double* C, const int* act) {
  int inst;
  if (!batch_on(act, inst)) return;
  A += (i64)inst * n; Bv += (i64)inst * n; C += (i64)inst * n;
  for (i64 x = (i64)blockIdx.x * blockDim.x + threadIdx.x; x < n; x += (i64)gridDim.x * blockDim.x)
    C[x] = A[x] * ax + Bv[x] * bx;
}
static unsigned stream_grid(i64 n) {
  i64 g = (n + 255) / 256;
  if (g > 8192) g = 8192;
  if (g < 1) g = 1;
  return (unsigned)g;
}

void launch_axpy(i64 n, const double* A, double ax, const double* Bv, double bx, double* C, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy, dim3(stream_grid(n)), dim3(256), 0, s, n, A, ax, Bv, bx, C, (const int*)nullptr);
}
// the same on ninst instances back to back (stride n), act-masked
void launch_axpy_b(i64 n, const double* A, double ax, const double* Bv, double bx, double* C, int ninst,
                   const int* act, hipStream_t s) {
  unsigned g = stream_grid(n);
  if (ninst > 1 && g > 1024) g = 1024;
  hipLaunchKernelGGL(k_axpy, dim3(g, ninst), dim3(256), 0, s, n, A, ax, Bv, bx, C, act);
}

// mat_frob_norm, basic_IMSRG.f90:4056-4087: weighted sum of squares per chunk
__global__ __launch_bounds__(256) void k_norm_partials(const double* op, const i64* coff, const int* clen,
                                                       const double* cw, double* part, i64 sop, i64 spart,
                                                       const int* act) {
  __shared__ double red[256];
  int inst;
  if (!batch_on(act, inst)) return;
  op += (i64)inst * sop;
  part += (i64)inst * spart;
  const int c = blockIdx.x;
  const double* x = op + coff[c];
  const int n = clen[c];
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) v += x[i] * x[i];
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) part[c] = s * cw[c];
}
// The tail of one nested commutator in one pass over its result T: lower
// triangles of the square blocks T(y, x) = herm T(x, y), X += c * T (E0 by
// task 0's first thread) and the norm partials of T (append_operator +
// mat_frob_norm, IMSRG_MAGNUS.f90:227-229).  Memory bound, and at small sizes
// the latency of one load -> LDS -> store chain: a task is a kTail x kTail
// tile pair of a square block (upper tile through LDS, every load issued
// before the barrier) or a run of at most kTailRun elements of T outside
// them.  Against symmetrising and then appending in a second pass: decoupling
// eMax 4 23.3 -> 21.6 ms, BCH eMax 6 (22O) 3.71 -> 3.42 ms, eMax 10 70.9 ->
// 70.1 ms; 32-wide tiles keep all loads of a thread in registers (51 VGPRs,
// 8 waves a SIMD).
__global__ __launch_bounds__(256) void k_comm_tail(DevBasis B, const TailTask* tasks, double* T, int herm, double* X,
                                                   double c, double* part) {
  __shared__ double S[kTail][kTail + 1];
  __shared__ double red[256];
  int inst;
  if (!batch_inst(B, inst)) return;
  X += (i64)inst * B.oplen;
  T += (i64)inst * B.oplen;
  part += (i64)inst * B.spart;
  const TailTask t = tasks[blockIdx.x];
  if (blockIdx.x == 0 && threadIdx.x == 0) X[0] = X[0] * 1.0 + T[0] * c;
  double v = 0.0;
  const int n = t.n;
  if (n > 0) {
    constexpr int C = kTail * kTail / 256;
    double* Tb = T + t.off;
    double* Xb = X + t.off;
    const int x0 = t.ti * kTail, y0 = t.tj * kTail;
    const int tx = threadIdx.x & (kTail - 1), ty = threadIdx.x / kTail;
    double a[C], u[C], w[C];
#pragma unroll
    for (int r = 0; r < C; ++r) {
      const int cl = ty + r * (256 / kTail);
      const int x = x0 + tx, y = y0 + cl, xl = y0 + tx, yl = x0 + cl;
      const bool in = x <= y && y < n, il = xl > yl && xl < n;   // x < n, yl < n follow
      a[r] = in ? Tb[x + (i64)y * n] : 0.0;
      u[r] = in ? Xb[x + (i64)y * n] : 0.0;
      w[r] = il ? Xb[xl + (i64)yl * n] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < C; ++r) S[ty + r * (256 / kTail)][tx] = a[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < C; ++r) {
      const int cl = ty + r * (256 / kTail);
      const int x = x0 + tx, y = y0 + cl, xl = y0 + tx, yl = x0 + cl;
      if (x <= y && y < n) {
        v += a[r] * a[r];
        Xb[x + (i64)y * n] = u[r] * 1.0 + a[r] * c;
      }
      if (xl > yl && xl < n) {
        const double b = herm * S[tx][cl];
        v += b * b;
        Tb[xl + (i64)yl * n] = b;
        Xb[xl + (i64)yl * n] = w[r] * 1.0 + b * c;
      }
    }
  } else {
    for (int i = threadIdx.x; i < t.ti; i += 256) {
      const double y = T[t.off + i];
      v += y * y;
      X[t.off + i] = X[t.off + i] * 1.0 + y * c;
    }
  }
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s * t.w;
}
void launch_comm_tail(const DevBasis& B, const TailTask* t, int nt, double* T, int herm, double* X, double c,
                      double* part, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_comm_tail, dim3(nt, B.ninst), dim3(256), 0, s, B, t, T, herm, X, c, part);
}

// X += c * T (every element, E0 by chunk 0's first thread) and the norm
// partials of T in the same pass: the axpy and norm of one nested
// commutator (append_operator + mat_frob_norm, IMSRG_MAGNUS.f90:227-229),
// each element's update and each chunk's partial sum exactly as k_axpy and
// k_norm_partials form them
__global__ __launch_bounds__(256) void k_axpy_norm(double* X, const double* T, double c, const i64* coff,
                                                   const int* clen, const double* cw, double* part, i64 sop, i64 spart,
                                                   const int* act) {
  __shared__ double red[256];
  int inst;
  if (!batch_on(act, inst)) return;
  X += (i64)inst * sop;
  T += (i64)inst * sop;
  part += (i64)inst * spart;
  const int ch = blockIdx.x;
  if (ch == 0 && threadIdx.x == 0) X[0] = X[0] * 1.0 + T[0] * c;
  const i64 o = coff[ch];
  const int n = clen[ch];
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const double y = T[o + i];
    v += y * y;
    X[o + i] = X[o + i] * 1.0 + y * c;
  }
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) part[ch] = s * cw[ch];
}
void launch_axpy_norm_b(const DevBasis& B, double* X, const double* T, double c, const i64* chunk_off,
                        const int* chunk_len, const double* chunk_w, int nchunk, double* part, hipStream_t s) {
  if (nchunk <= 0) return;
  hipLaunchKernelGGL(k_axpy_norm, dim3(nchunk, B.ninst), dim3(256), 0, s, X, T, c, chunk_off, chunk_len, chunk_w, part,
                     B.oplen, B.spart, B.act);
}

__global__ __launch_bounds__(1024) void k_sum_sqrt(const double* part, int n, double* dst, int do_sqrt, i64 spart,
                                                   i64 sdst, const int* act) {
  __shared__ double red[1024];
  int inst;
  if (!batch_on(act, inst)) return;
  part += (i64)inst * spart;
  dst += (i64)inst * sdst;
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) v += part[i];
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) dst[0] = do_sqrt ? sqrt(s) : s;
}

void launch_norm_partials_b(const DevBasis& B, const double* op, const i64* chunk_off, const int* chunk_len,
                            const double* chunk_w, int nchunk, double* part, hipStream_t s) {
  if (nchunk <= 0) return;
  hipLaunchKernelGGL(k_norm_partials, dim3(nchunk, B.ninst), dim3(256), 0, s, op, chunk_off, chunk_len, chunk_w, part,
                     B.oplen, B.spart, B.act);
}
void launch_sum_sqrt_b(const DevBasis& B, const double* part, int n, double* dst, i64 sdst, int do_sqrt,
                       hipStream_t s) {
  hipLaunchKernelGGL(k_sum_sqrt, dim3(1, B.ninst), dim3(1024), 0, s, part, n, dst, do_sqrt, B.spart, sdst, B.act);
}

// ======================================================== white generator
// twobody_monopole, basic_IMSRG.f90:2075-2090, for every orbit pair
__global__ __launch_bounds__(256) void k_monopole(DevBasis B, const double* H, double* M) {
  int inst;
  if (!batch_inst(B, inst)) return;
  H += (i64)inst * B.oplen;
  M += (i64)inst * B.N * B.N;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= B.N * B.N) return;
  const int a = idx % B.N, b = idx / B.N;
  const int ja = B.jj[a], jb = B.jj[b];
  double sm = 0.0;
  for (int JT = abs(ja - jb); JT <= ja + jb; JT += 2) sm = sm + (JT + 1) * v_elem(B, H, 1, a, b, a, b, JT);
  M[idx] = sm / (ja + 1.0) / (jb + 1.0);
}
void launch_monopole(const DevBasis& B, const double* H, double* M, hipStream_t s) {
  hipLaunchKernelGGL(k_monopole, dim3((B.N * B.N + 255) / 256, B.ninst), dim3(256), 0, s, B, H, M);
}

// Ground-state generators: the energy denominators of build_gs_white
// (generators.f90:4-106) from Hd, the numerators from Hn:
//   mode 0 (white, generators.f90:54,100):  eta = Hn / Eden
//   mode 1 (atan / atanxx, generators.f90:213,263 and 318,366):
//                                            eta = 0.5 atan(2 Hn / Eden)
// (build_gs_atan is mode 1 with Hd = Hn; build_gs_atanxx passes Hold as Hd)
__device__ __forceinline__ double gen_value(double x, double Eden, int mode) {
  return mode == 0 ? x / Eden : atan(2 * x / Eden) * 0.5;
}

// one-body part (also zeroes fhh, fpp)
__global__ __launch_bounds__(256) void k_gen_1b(DevBasis B, const double* Hd, const double* Hn, double* ETA,
                                                int mode) {
  int inst;
  if (!batch_inst(B, inst)) return;
  Hd += (i64)inst * B.oplen;
  Hn += (i64)inst * B.oplen;
  ETA += (i64)inst * B.oplen;
  const i64 idx = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  const i64 nA = (i64)B.A * B.A, nPA = (i64)B.P * B.A, nP = (i64)B.P * B.P;
  if (idx < nA) { ETA[B.off_fhh + idx] = 0.0; return; }
  if (idx < nA + nP) { ETA[B.off_fpp + (idx - nA)] = 0.0; return; }
  if (idx >= nA + nP + nPA) return;
  const i64 x = idx - nA - nP;
  const int a = (int)(x % B.P), i = (int)(x / B.P);
  const int ak = B.parts[a], ik = B.holes[i];
  if (B.jj[ik] != B.jj[ak] || B.ll[ik] != B.ll[ak] || B.tz[ik] != B.tz[ak]) return;
  const int ji = B.jj[ik];
  double Eden = 0.0;
  for (int JT = 0; JT <= 2 * ji; JT += 2) Eden = Eden - (JT + 1) * v_elem(B, Hd, 1, ak, ik, ak, ik, JT);
  Eden = Eden / (ji + 1.0) / (ji + 1.0);
  Eden = Eden + Hd[B.off_fpp + a + (i64)a * B.P] - Hd[B.off_fhh + i + (i64)i * B.A];
  ETA[B.off_fph + x] = gen_value(Hn[B.off_fph + x], Eden, mode);
}
void launch_gen_1b(const DevBasis& B, const double* Hd, const double* Hn, double* ETA, int mode, hipStream_t s) {
  const i64 n = (i64)B.A * B.A + (i64)B.P * B.P + (i64)B.P * B.A;
  hipLaunchKernelGGL(k_gen_1b, dim3((unsigned)((n + 255) / 256), B.ninst), dim3(256), 0, s, B, Hd, Hn, ETA, mode);
}

// two-body part, full-segment tasks (gam3 from the formula, the rest zero);
// M = the monopoles of Hd
__global__ __launch_bounds__(256) void k_gen_2b(DevBasis B, const SegTask* tasks, const double* Hd, const double* M,
                                                const double* Hn, double* ETA, int mode) {
  int inst;
  if (!batch_inst(B, inst)) return;
  Hd += (i64)inst * B.oplen;
  Hn += (i64)inst * B.oplen;
  ETA += (i64)inst * B.oplen;
  M += (i64)inst * B.N * B.N;
  const SegTask t = tasks[blockIdx.x];
  const i64 e = (i64)t.start + threadIdx.x;
  if (e >= t.cnt) return;
  const int q = t.q, g = t.g;
  const i64 o = B.goff[q * 6 + g] + e;
  if (g != 2) { ETA[o] = 0.0; return; }
  const int np = B.dims[q * 3];
  const int IX = (int)(e % np), JX = (int)(e / np);
  int a, b, i, j;
  unpack(B.pairs[B.pairoff[q * 3 + 0] + IX], a, b);
  unpack(B.pairs[B.pairoff[q * 3 + 2] + JX], i, j);
  const int N = B.N;
  double Eden = 0.0;
  Eden = Eden + M[a + b * N];
  Eden = Eden + M[i + j * N];
  Eden = Eden - M[a + i * N];
  Eden = Eden - M[a + j * N];
  Eden = Eden - M[i + b * N];
  Eden = Eden - M[j + b * N];
  Eden = Eden + f_elem(B, Hd, 1, a, a) + f_elem(B, Hd, 1, b, b) - f_elem(B, Hd, 1, i, i) - f_elem(B, Hd, 1, j, j);
  ETA[o] = gen_value(Hn[o], Eden, mode);
}
void launch_gen_2b(const DevBasis& B, const SegTask* t, int nt, const double* Hd, const double* M, const double* Hn,
                   double* ETA, int mode, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_gen_2b, dim3(nt, B.ninst), dim3(256), 0, s, B, t, Hd, M, Hn, ETA, mode);
}

// mbpt2, basic_IMSRG.f90:4165-4199: one partial per gam3 tile
__global__ __launch_bounds__(256) void k_mbpt2_partials(DevBasis B, const SegTask* tasks, const double* H,
                                                        double* part) {
  int inst;
  if (!batch_inst(B, inst)) return;
  H += (i64)inst * B.oplen;
  part += (i64)inst * B.spart;
  __shared__ double red[256];
  const SegTask t = tasks[blockIdx.x];
  const i64 e = (i64)t.start + threadIdx.x;
  double v = 0.0;
  const int q = t.q;
  if (e < t.cnt) {
    const int np = B.dims[q * 3];
    const int II = (int)(e % np), JJ = (int)(e / np);
    int i, j, k, l;
    unpack(B.pairs[B.pairoff[q * 3 + 0] + II], i, j);
    unpack(B.pairs[B.pairoff[q * 3 + 2] + JJ], k, l);
    const double fi = f_elem(B, H, 1, i, i), fj = f_elem(B, H, 1, j, j);
    const double fk = f_elem(B, H, 1, k, k), fl = f_elem(B, H, 1, l, l);
    const double eden = fk + fl - fi - fj;
    const double x = H[B.goff[q * 6 + 2] + e];
    v = x * x / eden;
  }
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s * (B.chJ[q] + 1.0);
}
void launch_mbpt2_partials(const DevBasis& B, const SegTask* t, int nt, const double* H, double* part,
                           hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_mbpt2_partials, dim3(nt, B.ninst), dim3(256), 0, s, B, t, H, part);
}

// ============================================================ normal_order
// basic_IMSRG.f90:2419-2550.  scratch[0] receives E0; then the one-body
// corrections are applied in place (every thread reads only the element it
// writes, so the in-place update equals the reference's TEMP copy).
__global__ __launch_bounds__(256) void k_no_e0(DevBasis B, const double* H, double* E0) {
  __shared__ double red[256];
  double v = 0.0;
  // 2 * sum_h f_hh (2j+1)
  for (int i = threadIdx.x; i < B.N; i += blockDim.x)
    if (B.con[i] == 1) v += f_elem(B, H, 1, i, i) * (B.jj[i] + 1);
  double s1 = block_sum(v, red) * 2.0;
  v = 0.0;
  for (int x = threadIdx.x; x < B.N * B.N; x += blockDim.x) {
    const int i = x / B.N, j = x % B.N;
    if (B.con[i] * B.con[j] == 0) continue;
    for (int JT = abs(B.jj[i] - B.jj[j]); JT <= B.jj[i] + B.jj[j]; JT += 2)
      v += v_elem(B, H, 1, i, j, i, j, JT) * (JT + 1);
  }
  const double s2 = block_sum(v, red);
  if (threadIdx.x == 0) E0[0] = (s1 + s2) * 0.5;
}

__global__ __launch_bounds__(256) void k_no_1b(DevBasis B, double* H) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= B.N * B.N) return;
  const int ax = idx % B.N, bx = idx / B.N;
  if (B.jj[ax] != B.jj[bx] || B.ll[ax] != B.ll[bx] || B.tz[ax] != B.tz[bx]) return;
  const int ca = B.con[ax], cb = B.con[bx];
  // the reference visits hh (a<=b), ph (a particle, b hole), pp (a<=b)
  if (ca == 1 && cb == 1 && B.cidx[ax] > B.cidx[bx]) return;
  if (ca == 0 && cb == 0 && B.cidx[ax] > B.cidx[bx]) return;
  if (ca == 1 && cb == 0) return;
  double sm = 0.0;
  for (int ix = 0; ix < B.N; ++ix) {
    if (B.con[ix] != 1) continue;
    for (int JT = abs(B.jj[ix] - B.jj[ax]); JT <= B.jj[ix] + B.jj[ax]; JT += 2)
      sm = sm + (JT + 1.0) / (B.jj[ax] + 1) * v_elem(B, H, 1, ax, ix, bx, ix, JT);
  }
  const double v = f_elem(B, H, 1, ax, bx) + sm;
  const int a = B.cidx[ax], b = B.cidx[bx];
  if (ca == 1) {
    H[B.off_fhh + a + (i64)b * B.A] = v;
    H[B.off_fhh + b + (i64)a * B.A] = v;
  } else if (cb == 1) {
    H[B.off_fph + a + (i64)b * B.P] = v;
  } else {
    H[B.off_fpp + a + (i64)b * B.P] = v;
    H[B.off_fpp + b + (i64)a * B.P] = v;
  }
}

__global__ void k_set_e0(double* H, const double* E0) { H[0] = E0[0]; }

// vectorize / repackage, basic_IMSRG.f90:3929-4053: one workgroup per run.
// In repackage the lower element X(j,i) is stored before its partner
// X(i,j) = herm * v by the same thread, so a diagonal element ends as
// herm * v, as in the reference's loop.
__global__ __launch_bounds__(256) void k_vectorize(const VecTask* tasks, double* op, double* vec, int dir,
                                                   double herm) {
  const VecTask t = tasks[blockIdx.x];
  for (int x = threadIdx.x; x < t.len; x += blockDim.x) {
    if (dir == 0) {
      vec[t.vec_off + x] = op[t.op_off + x];
    } else {
      const double v = vec[t.vec_off + x];
      op[t.op_off + x] = v;
      if (t.mirror) op[t.op_off + (i64)x * t.mirror] = v * herm;
    }
  }
}
void launch_vectorize(const VecTask* t, int nt, double* op, double* vec, int dir, int herm, hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_vectorize, dim3(nt), dim3(256), 0, s, t, op, vec, dir, (double)herm);
}

// E0 = v for every instance of an operator array
__global__ void k_fill_e0(DevBasis B, double* op, double v) {
  int inst;
  if (!batch_inst(B, inst)) return;
  if (threadIdx.x == 0) op[(i64)inst * B.oplen] = v;
}
void launch_fill_e0(const DevBasis& B, double* op, double v, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_e0, dim3(1, B.ninst), dim3(64), 0, s, B, op, v);
}

void launch_normal_order(const DevBasis& B, double* H, double* scratch, hipStream_t s) {
  hipLaunchKernelGGL(k_no_e0, dim3(1), dim3(256), 0, s, B, H, scratch);
  hipLaunchKernelGGL(k_no_1b, dim3((B.N * B.N + 255) / 256), dim3(256), 0, s, B, H);
  hipLaunchKernelGGL(k_set_e0, dim3(1), dim3(1), 0, s, H, scratch);
}

// ================================================================ helpers
__global__ void k_fill(double* p, i64 n, double v, const int* act) {
  int inst;
  if (!batch_on(act, inst)) return;
  p += (i64)inst * n;
  for (i64 x = (i64)blockIdx.x * blockDim.x + threadIdx.x; x < n; x += (i64)gridDim.x * blockDim.x) p[x] = v;
}
__global__ void k_copy(double* d, const double* s, i64 n, const int* act) {
  int inst;
  if (!batch_on(act, inst)) return;
  d += (i64)inst * n;
  s += (i64)inst * n;
  for (i64 x = (i64)blockIdx.x * blockDim.x + threadIdx.x; x < n; x += (i64)gridDim.x * blockDim.x) d[x] = s[x];
}
void launch_fill(double* p, i64 n, double v, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill, dim3(stream_grid(n)), dim3(256), 0, s, p, n, v, (const int*)nullptr);
}
void launch_copy(double* dst, const double* src, i64 n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_copy, dim3(stream_grid(n)), dim3(256), 0, s, dst, src, n, (const int*)nullptr);
}
void launch_fill_b(double* p, i64 n, double v, int ninst, const int* act, hipStream_t s) {
  if (n <= 0) return;
  unsigned g = stream_grid(n);
  if (ninst > 1 && g > 1024) g = 1024;
  hipLaunchKernelGGL(k_fill, dim3(g, ninst), dim3(256), 0, s, p, n, v, act);
}
void launch_copy_b(double* dst, const double* src, i64 n, int ninst, const int* act, hipStream_t s) {
  if (n <= 0) return;
  unsigned g = stream_grid(n);
  if (ninst > 1 && g > 1024) g = 1024;
  hipLaunchKernelGGL(k_copy, dim3(g, ninst), dim3(256), 0, s, dst, src, n, act);
}

// ====================================================== transform_2b_to_HF
// HF_mod.f90:567-692: each channel's two-body blocks as one square matrix
// over its pairs in the order (hh, ph, pp), nt x nt column-major at
// V + voff[q] (square blocks as stored, rectangular blocks in both
// orientations); unpack writes the six blocks back from it.  One thread per
// stored element (the full-block segment tasks).
__device__ __forceinline__ void hf_pos(const DevBasis& B, int q, int g, i64 e, int& n1, i64& row, i64& col, i64& nt) {
  const int np = B.dims[q * 3], nb = B.dims[q * 3 + 1], nh = B.dims[q * 3 + 2];
  const int r0[3] = {nh + nb, nh, 0};
  n1 = brows(B, q, g);
  row = r0[row_cls(g)] + e % n1;
  col = r0[col_cls(g)] + e / n1;
  nt = (i64)np + nb + nh;
}

__global__ __launch_bounds__(256) void k_hf_pack(DevBasis B, const SegTask* tasks, const double* op, double* V,
                                                 const i64* voff) {
  const SegTask t = tasks[blockIdx.x];
  const i64 e = (i64)t.start + threadIdx.x;
  if (e >= t.cnt) return;
  int n1;
  i64 row, col, nt;
  hf_pos(B, t.q, t.g, e, n1, row, col, nt);
  const double x = op[B.goff[t.q * 6 + t.g] + e];
  double* Vq = V + voff[t.q];
  Vq[row + col * nt] = x;
  if (!is_square(t.g)) Vq[col + row * nt] = x;
}

__global__ __launch_bounds__(256) void k_hf_unpack(DevBasis B, const SegTask* tasks, const double* V,
                                                   const i64* voff, double* op) {
  const SegTask t = tasks[blockIdx.x];
  const i64 e = (i64)t.start + threadIdx.x;
  if (e >= t.cnt) return;
  int n1;
  i64 row, col, nt;
  hf_pos(B, t.q, t.g, e, n1, row, col, nt);
  op[B.goff[t.q * 6 + t.g] + e] = V[voff[t.q] + row + col * nt];
}

void launch_hf_pack(const DevBasis& B, const SegTask* t, int nt, const double* op, double* V, const i64* voff,
                    hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_hf_pack, dim3(nt), dim3(kTile), 0, s, B, t, op, V, voff);
}

void launch_hf_unpack(const DevBasis& B, const SegTask* t, int nt, const double* V, const i64* voff, double* op,
                      hipStream_t s) {
  if (nt <= 0) return;
  hipLaunchKernelGGL(k_hf_unpack, dim3(nt), dim3(kTile), 0, s, B, t, V, voff, op);
}

// ==================================== a small commutator in three launches
// At eMax <= 4 every term kernel of the fused commutator lasts 4 - 13 us, a
// few dependent memory latencies, and a graph of fourteen of them with joins
// between queues spends as long between kernels as in them.  Here the terms
// that do not wait for each other share a launch, one range of workgroups
// each, the longest first: the bodies, and so the sums, are those of the
// separate kernels.  Decoupling eMax 4 (174 nested commutators) 20.5 -> 10.6 ms.
// Larger bases fill the chip term by term and take kernels that do not fit
// here (register-direct tiles, block quadruples).
union PhaseLds {
  GemmLds<32, 32> g;
  double s[64][65];
  double f[64 * 65];
};

template <int SIG>
__device__ __forceinline__ void phase_gemm(PhaseLds& lds, const PhaseGemm& f, int bx) {
  const int ti = xcd_task(f.xm, bx);
  if (ti < 0 || ti >= f.n) return;   // the range is rounded up
  gemm_tile<32, 32, SIG>(lds.g, f.sl, f.probs, f.tasks[ti], blockIdx.y, f.as, f.s2);
}

__global__ __launch_bounds__(256) void k_phase1(DevBasis B, Phase1 P) {
  __shared__ PhaseLds lds;
  int inst;
  if (!batch_inst(B, inst)) return;
  int b = blockIdx.x;
  if (b < P.k2.grid) return phase_gemm<0>(lds, P.k2, b);
  b -= P.k2.grid;
  if (b < P.pp1.grid) return phase_gemm<8>(lds, P.pp1, b);
  b -= P.pp1.grid;
  if (b < P.k3.grid) return phase_gemm<1>(lds, P.k3, b);
  b -= P.k3.grid;
  if (b < P.g122) {
    if (b < P.n122)
      d_comm122p(B, P.seg, P.part, P.partT, P.pstride, P.rowp, P.colp, P.f1off, P.nf1, P.L, P.Lh, P.R, P.Rh, P.RES,
                 P.RESh, 0, b, P.n122, lds.f);
    return;
  }
  b -= P.g122;
  if (b < P.gcc) {
    if (b < P.ncc) d_pandya(B, P.cc, P.R, P.Rh, P.RCC, b, P.ncc);
    return;
  }
  b -= P.gcc;
  if (b < P.n111) return d_comm111(B, P.L, P.Lh, P.R, P.Rh, P.RES, b);
  b -= P.n111;
  d_e0_partials(B, P.L, P.Lh, P.R, P.Rh, P.epart, b, lds.f);
}

__global__ __launch_bounds__(256) void k_phase2(DevBasis B, Phase2 P) {
  __shared__ PhaseLds lds;
  int inst;
  if (!batch_inst(B, inst)) return;
  int b = blockIdx.x;
  if (b < P.ph.grid) return phase_gemm<10>(lds, P.ph, b);
  b -= P.ph.grid;
  if (b < P.npairs) return d_pppp_sym1(B, P.pairs, P.RES, P.w1, P.Lh * P.Rh, 1, b, lds.s);
  b -= P.npairs;
  if (b < P.nepi)
    return d_pphh_epilogue(B, P.epi, P.L, P.Lh, P.R, P.Rh, P.RES, P.w1, P.w2, P.Pscr, P.poff, P.k3ks, P.K2scr,
                           P.k2off, P.k2ks, b);
  d_e0_final(P.epart, B.nblocks, P.Lh * P.Rh == -1 ? 1 : 0, 1, P.RES, 0, B.spart, B.oplen, B.act, lds.f);
}

// 121 and 221 of a one-body element in its workgroup, in that order
__global__ __launch_bounds__(512) void k_phase3(DevBasis B, Phase3 P) {
  __shared__ union { PhChunkLds c; double red[kOneLanes]; } lds;
  int inst;
  if (!batch_inst(B, inst)) return;
  int b = blockIdx.x;
  if (b < P.g1) {
    if (b >= P.none) return;
    d_comm121(B, P.one, P.L, P.Lh, P.R, P.Rh, P.RES, P.RESh, b, lds.red);
    __syncthreads();
    d_comm221(B, P.one, P.L, P.Lh, P.R, P.Rh, P.w1, P.w2, P.RES, P.RESh, b, lds.red);
    return;
  }
  b -= P.g1;
  d_comm222ph_chunk(B, P.phc, P.fq, P.fql, P.fqi, P.quad, P.WCC, P.Lh, P.Rh, P.RES, P.RESh, 0, b, P.nphc, lds.c);
}

bool launch_phase1(const DevBasis& B, Phase1 P, int e0, hipStream_t s) {
  if (2 * P.nf1 * sizeof(double) > sizeof(PhaseLds)) return false;
  const i64 n = (i64)B.A * B.A + (i64)B.P * B.A + (i64)B.P * B.P;
  auto up = [](int x) { return (x + kXcds - 1) / kXcds * kXcds; };   // ranges start on XCD 0, as the task orders assume
  P.k2.grid = up(P.k2.grid); P.pp1.grid = up(P.pp1.grid); P.k3.grid = up(P.k3.grid);
  P.g122 = up(P.n122); P.gcc = up(P.ncc);
  P.n111 = (int)((n + 3) / 4);
  const int grid = P.k2.grid + P.pp1.grid + P.k3.grid + P.g122 + P.gcc + P.n111 + (e0 ? B.nblocks + 1 : 0);
  if (grid > 0) hipLaunchKernelGGL(k_phase1, dim3(grid, B.ninst), dim3(256), 0, s, B, P);
  return true;
}
void launch_phase2(const DevBasis& B, Phase2 P, int e0, hipStream_t s) {
  P.ph.grid = (P.ph.grid + kXcds - 1) / kXcds * kXcds;
  const int grid = P.ph.grid + P.npairs + P.nepi + (e0 ? 1 : 0);
  if (grid > 0) hipLaunchKernelGGL(k_phase2, dim3(grid, B.ninst), dim3(256), 0, s, B, P);
}
void launch_phase3(const DevBasis& B, Phase3 P, hipStream_t s) {
  P.g1 = (P.none + kXcds - 1) / kXcds * kXcds;
  const int grid = P.g1 + P.nphc;
  if (grid > 0) hipLaunchKernelGGL(k_phase3, dim3(grid, B.ninst), dim3(512), 0, s, B, P);
}

}  // namespace imsrg
