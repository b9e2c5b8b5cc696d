// Tensor operators (rank > 0) on the device: layout tables and the kernels of
// the scalar-tensor commutator [L, R] (L scalar, R a tensor of rank
// lambda = rank/2 and parity change dpar/2), TS_commutators.f90:10-1849.
//
// Flat tensor layout (allocate_tensor, basic_IMSRG.f90:688-951):
//   [E0 | fhh (A x A) | fph (P x A) | fpp (P x P) | per block q:
//    tgam1..tgam9, tgam g = (pairs of class sea1(g) in channel (J1,Tz,P1)) x
//    (pairs of class sea2(g) in channel (J2,Tz,P2)), column-major]
// blocks in the reference's loop order (2J1 outer, 2J2 = max(|2J1 - rank|,
// 2J1) .. 2J1 + rank, Tz = -1..1, P1 = 0..1); blocks with 2J2 > 2 jmax are
// empty.  The one-body offsets are the scalar operator's.
#pragma once

#include "basis.hpp"
#include "kernels.hpp"

namespace imsrg {

// pair class (0 pp, 1 ph, 2 hh) of the rows / columns of tgam g (sea1 / sea2,
// basic_IMSRG.f90:127)
constexpr int kTSea1[9] = {0, 0, 0, 1, 2, 1, 2, 1, 2};
constexpr int kTSea2[9] = {0, 1, 2, 1, 2, 2, 0, 0, 1};

struct DevTensor {
  int rank, dpar, nblocks, ncc;
  i64 oplen, off2b;                // doubles of an operator; first two-body element
  const int* blk;                  // [nblocks*8] 2J1 2J2 Tz P1 P2 q1 q2 -
  const int* tdim;                 // [nblocks*6] np1 nb1 nh1 np2 nb2 nh2
  const i64* tgoff;                // [nblocks*9]
  const int* look;                 // [((2J1/2)*(rank/2+1) + (2J2-2J1)/2)*6 + 2(Tz+1) + P1] -> q
  const int* cblk;                 // [ncc*8] 2J3 2J4 Tz PAR r1 r2 nb1 nb2
  const int* cscal;                // [ncc*2] scalar cross-coupled blocks of the rows (J3) and columns (J4)
  const i64* coff;                 // [ncc*3] CCX, CCR, W offsets
  const int* cclook;               // [(2J3/2)*(rank/2+1) + (2J4-2J3)/2] -> qx of (J3, J4, Tz 0, PAR 0)
  const double* x6;                // {J1 J2 rank; j4 j5 j6}: [J1/2][J2/2][j4/2][j5/2][j6/2]
  const double* s6;                // {c d J2; b x J4}:       [c/2][d/2][b/2][x/2][J2/2][J4/2]
  const i64* wtab;                 // [(((2J3/2)*(rank/2+1) + (2J4-2J3)/2)*4 + 2 Tz + PAR)*2]: offset of the
                                   // product W of that cross-coupled block, its leading dimension
  const double* n9;                // 9j {u1 u2 J3; u4 u5 J4; J1 J2 rank} * sqrt((J3+1)(J4+1)) of the
                                   // 222_ph back-transform, J3 <= J4 <= J3 + rank, J1 <= J2 <= J1 + rank:
                                   // [u1/2][u2/2][u4/2][u5/2][J3/2][(J4-J3)/2][J1/2][(J2-J1)/2]
                                   // (the outputs of one orbit quadruple read one contiguous run)
  const int *fst, *fmem;           // orbits of 2j = 2j_x - rank + 2r that a rank / dpar one-body operator couples
                                   // to orbit x: fmem[fst[k]] .. fmem[fst[k + 1] - 1], k = x (rank + 1) + r
  int nJ, nhx, nho;                // 2J/2 values; half-integers up to jmax + rank; up to jmax
};

// one sub-block g of block q and its pair lists
struct TSub { int q, g, n1, n2; i64 off, roff, coff; };
// 256 consecutive elements of sub-block sb
struct TElem { int sb; int start; };
// one output element of the 222_ph back-transform: its offset, its orbits
// (a | b << 8 | c << 16 | d << 24) and 2J1 | 2J2 << 16; the list is ordered
// by orbit quadruple, so the lanes of a wave share the quadruple's loops
struct TPh { int off, abcd, jj; };
// at most 64 quadruples of that list (quads q0 .. q0 + nq: orbits, first
// output) with the same four j, patterns and outputs (J1, J2)
struct TPack { int q0, nq, no; unsigned mask; };
// 212 and 222_ph run by packs from kTsPackMin orbit quadruples on, below by one
// thread per output: a pack's wave runs through its terms one after the other,
// so few packs (about nq / 50) leave the chip waiting, however many outputs a
// quadruple has.  Whole commutator, us, by output / by packs: eMax 4 rank 8 (33 k
// quadruples) 820 / 1565, eMax 5 rank 0 (122 k) 386 / 395, rank 4 (135 k) 1327 / 1404,
// rank 8 (128 k, 888 k outputs) 1826 / 2411; eMax 14 lMax 1 rank 2 (180 k) 569 / 510,
// eMax 6 rank 0 (376 k) 754 / 665, rank 4 (415 k) 3620 / 2971, eMax 7 lMax 5 rank 4
// (727 k) 6428 / 3921.
constexpr i64 kTsPackMin = 160000;
constexpr int kTsOut = 16;    // outputs a lane accumulates at a time
constexpr int kTsRows = 64;   // (J3, J4) pairs whose coefficients are staged at a time

// The sixteen (case, target) forms of 222_ph's back-transform (tensor.hip):
// places of a, b, c, d among the output's orbits, and what a form needs
constexpr unsigned pos4(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }
constexpr unsigned long long pos8(unsigned a, unsigned b, unsigned c, unsigned d, unsigned e, unsigned f, unsigned g,
                                  unsigned h) {
  return (unsigned long long)(a | (b << 8) | (c << 16) | (d << 24)) |
         ((unsigned long long)(e | (f << 8) | (g << 16) | (h << 24)) << 32);
}
constexpr unsigned long long kPatPos0 = pos8(pos4(0, 1, 2, 3), pos4(2, 3, 0, 1), pos4(0, 1, 3, 2), pos4(2, 3, 1, 0),
                                             pos4(1, 0, 2, 3), pos4(3, 2, 0, 1), pos4(1, 0, 3, 2), pos4(3, 2, 1, 0));
constexpr unsigned long long kPatPos1 = pos8(pos4(3, 1, 2, 0), pos4(1, 3, 0, 2), pos4(2, 1, 3, 0), pos4(0, 3, 1, 2),
                                             pos4(3, 0, 2, 1), pos4(1, 2, 0, 3), pos4(2, 0, 3, 1), pos4(0, 2, 1, 3));
constexpr unsigned kPatBra = 0xd8d8, kPatKet = 0xe4e4, kPat34 = 0xaa55;   // kPat34: sign (-1)^((J3+J4)/2)

struct TPat { int a, b, c, d; };
__host__ __device__ inline TPat ts_pat(int pat, int u) {
  const unsigned m = (unsigned)((pat < 8 ? kPatPos0 : kPatPos1) >> (8 * (pat & 7))) & 255;
  TPat x;
  x.a = (u >> (8 * (m & 3))) & 255;
  x.b = (u >> (8 * ((m >> 2) & 3))) & 255;
  x.c = (u >> (8 * ((m >> 4) & 3))) & 255;
  x.d = (u >> (8 * ((m >> 6) & 3))) & 255;
  return x;
}

// one-body output: cls 0 fhh (p <= q, mirrored), 1 fpp (p <= q, mirrored), 2 fph
struct TOne { int cls, p, q, pad; };
// 256 consecutive elements of CCX (term 1) or CCR (term 2) of block qx
struct TCC { int qx, term, start, pad; };

void launch_ts111(const DevBasis& B, const DevTensor& T, const double* L, int Lh, const double* R, int Rh,
                  double* RES, hipStream_t s);
// mode 0: TS_commutator_121, 1: TS_commutator_211 (X = the scalar
// cross-coupled set of L), 2: TS_commutator_221 (X = w1, Y = w2, pm = Lh)
void launch_ts_one(int mode, const DevBasis& B, const DevTensor& T, const TOne* t, int nt, const double* L, int Lh,
                   const double* X, const double* Y, const double* R, int Rh, double* RES, int RESh, hipStream_t s);
// TS_commutator_122 (assigns) over element tiles
void launch_ts122(const DevBasis& B, const DevTensor& T, const TSub* sb, const TElem* t, int nt, const double* L,
                  int Lh, const double* R, int Rh, double* RES, hipStream_t s);
// TS_commutator_212 (adds)
void launch_ts212(const DevBasis& B, const DevTensor& T, const TPh* t, i64 nt, const TPack* p, int np, const int2* q,
                  const double* L, int Lh, const double* R, int Rh, double* RES, hipStream_t s);
// the back-transform of TS_commutator_222_ph from the products Wx / Wy
void launch_ts_ph(const DevBasis& B, const DevTensor& T, const TPh* t, i64 nt, const TPack* p, int np, const int2* q,
                  int Lh, int Rh, const double* Wx, const double* Wy, double* RES, hipStream_t s);
// calculate_single_pandya of every listed (block, term) into CC
void launch_ts_pandya(const DevBasis& B, const DevTensor& T, const TCC* t, int nt, const double* R, int Rh,
                      double* CC, hipStream_t s);
// RES[x] += w1[x] - w2[x] over [off, off + n)
void launch_ts_epilogue(i64 off, i64 n, const double* w1, const double* w2, double* RES, hipStream_t s);
// weighted sum of squares over segments (off, len, weight): part[k] per
// chunk k of 4096 elements (chunk table ck: segment offset, length, weight),
// then dst = sqrt(sum part) in chunk order
void launch_wnorm(const i64* ck_off, const int* ck_len, const double* ck_w, int nck, const double* op, double* part,
                  double* dst, hipStream_t s);

}  // namespace imsrg
