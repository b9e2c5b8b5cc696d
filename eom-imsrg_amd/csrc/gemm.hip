// Grouped FP64 MFMA GEMM for gfx950 (v_mfma_f64_16x16x4f64).
//
// One launch runs a list of tile tasks over a list of problems
//   C = alpha * (op(A1) op(B1) + s2 * op(A2) op(B2))  (+ beta C),
// operands addressed as (slot, offset) so a plan serves every call.  Tile
// shapes 64x64, 128x64, 128x128, 64x32, 32x64, 32x32 (256 threads = 4 waves
// in 2 x 2, each wave a (TBM/2) x (TBN/2) block of 16x16 MFMA tiles; the
// small shapes cut the edge padding of thin problems), K in steps of 16 through
// two LDS buffers with the next K-tile prefetched into registers; or (shapes
// 128x64 and 64x64 register-direct) each wave loading its own operands
// into registers with no LDS.  Split K:
// task.ks selects K-chunk [ks*kchunk, (ks+1)*kchunk) and slab C + ks*cstride.
#include <hip/hip_runtime.h>

#include "gemm_tile.hpp"

namespace imsrg {

namespace {

template <int TBM, int TBN, int SIG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(
    TBM * TBN <= 32 * 32 ? 8 : (TBM * TBN <= 64 * 64 ? 4 : (TBM * TBN <= 128 * 64 ? 2 : 1))))) void k_gemm_t(Slots sl, const GemmProb* probs, const GemmTask* tasks, XcdMap xm,
                                                double ascale, double s2scale) {
  __shared__ GemmLds<TBM, TBN> lds;
  const int ti = xcd_task(xm, blockIdx.x);
  if (ti < 0) return;
  int inst;
  if (!batch_on(sl.act, inst)) return;
  gemm_tile<TBM, TBN, SIG>(lds, sl, probs, tasks[ti], inst, ascale, s2scale);
}

// ------------------------------------------------------------------------
// Register-direct variant (tile shapes 6 and 7): the four waves of a
// workgroup compute independent WM x WN blocks of a (2 WM) x (2 WN) tile,
// each loading its MFMA operands from global memory straight into
// registers, kStages chunks of 8 k in flight; no LDS and no barriers.
// MFMA tiles 2p and 2p + 1 of a block hold its rows (columns) 32p + 2i and
// 32p + 2i + 1, i = lane % 16: an operand contiguous in its row / column
// index is one 16-byte load for both tiles, as is one contiguous in k for
// its two k of a chunk (buffer loads take any 8-byte alignment), and results
// leave in 16-byte stores.  Blocks that the matrix's edge cuts run a loop of
// their own with loads at clamped rows, so the loop of the whole blocks has
// no branch and no select: the address unit, busy 59 % of the
// time on W' and 71 % on PPPP (eMax 10) with 8-byte loads and clamps, was
// what kept the matrix cores at 50 % and 69 %.  Measured (us, before /
// now): PPPP eMax 8 131 / 106, 9 476 / 346, 10 1204 / 1030 (59 TFLOP/s); W'
// eMax 8 102 / 74, 9 273 / 204, 10 548 / 439; pp x (ph|hh) eMax 10 308 / 248.
// Two stages and two waves a SIMD: three stages 110 and 1020 (PPPP eMax 8,
// 10), three waves (spills) 130 and 1194.
constexpr int kStages = 2;
typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v2u __attribute__((ext_vector_type(2), aligned(8)));   // any 8-byte alignment

// one product of a wave: scale op(A)[m0:, k0:k1] op(B)[k0:k1, n0:]; the
// transposes are uniform run-time values where TT < 0
struct DProd {
  const double* A;
  const double* B;
  int lda, ldb, ta, tb, k0, k1;
  double scale;
};

// One operand of a wave: T MFMA tiles of rows (columns), its stages of
// fragments f[tile][MFMA of the chunk].  Buffer loads: a uniform base and
// uniform offset, so a lane holds 32-bit offsets only.  kin: contiguous in k.
// IL: tiles 2p and 2p + 1 hold every other row of 32 (else 16 rows each).
typedef unsigned v4w __attribute__((ext_vector_type(4)));
typedef unsigned v2w __attribute__((ext_vector_type(2)));
template <int T, int S, bool IL>
struct DOperand {
  double f[S][T][2];
  __amdgpu_buffer_rsrc_t rs;
  int ld, lim;       // lim: rows (columns) from the block's first to the matrix's end
  unsigned s0;       // byte offset of the next chunk (an operand stays below 4 GiB)
  int o, sh;         // lane offset in whole blocks; rows the base was moved back by

  static __device__ __forceinline__ int tr(int t) { return IL ? 32 * (t / 2) + (t & 1) : 16 * t; }
  __device__ __forceinline__ void set(const double* X, int r0, int k0, int l, bool kin, bool alt, int lim_, int lr,
                                      int kq) {
    ld = l;
    lim = lim_;
    s0 = 0;
    // pairs of rows: a block of one row starts at the row before (offsets are
    // unsigned, and the matrix has at least two rows)
    sh = !kin && lim == 1 ? 1 : 0;
    const uint64_t u = reinterpret_cast<uint64_t>(X + (kin ? (i64)r0 * l + k0 : r0 - sh + (i64)k0 * l));
    const uint64_t p = ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32) |
                       (unsigned)__builtin_amdgcn_readfirstlane((int)u);
    rs = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(p), 0, -1, 0x00020000);
    const int kk = alt ? kq : 2 * kq;
    o = 8 * (kin ? (IL ? 2 : 1) * lr * l + kk : 2 * lr + kk * l);
  }
  // lane offset of tile t's row in a block that the matrix's edge cuts: its
  // last row instead of rows beyond (their products are not stored)
  __device__ __forceinline__ int row(int t, bool kin, int lr) const {
    const int r = min(tr(t) + (IL ? 2 : 1) * lr, lim - 1);
    return 8 * (kin ? r * ld : r + sh);
  }
  __device__ __forceinline__ v2d ld2(int vo, unsigned so) const {
    const v4w x = __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so, 0);
    return __builtin_bit_cast(v2d, x);
  }
  __device__ __forceinline__ double ld1(int vo, unsigned so) const {
    const v2w x = __builtin_amdgcn_raw_buffer_load_b64(rs, vo, so, 0);
    return __builtin_bit_cast(double, x);
  }
  template <bool EDGE>
  __device__ __forceinline__ void load(int st, bool kin, bool alt, int lr, int kq) {
    if (kin) {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const v2d x = EDGE ? ld2(row(t, kin, lr) + 16 * kq, s0) : ld2(o, s0 + 8 * tr(t) * ld);
        f[st][t][0] = x[0];
        f[st][t][1] = x[1];
      }
      s0 += 64;
      return;
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const unsigned sg = s0 + 8 * g * (alt ? 4 : 1) * ld;
#pragma unroll
      for (int t = 0; t < T; t += 2) {
        // the pair of rows from 32 (t / 2) + 2 lr, in an edge block moved back
        // where it would pass the last row
        const v2d x = EDGE ? ld2(8 * (min(16 * t + 2 * lr, lim - 2) + sh + (alt ? kq : 2 * kq) * ld), sg)
                           : ld2(o + 128 * t, sg);
        f[st][t][g] = x[0];
        f[st][t + 1][g] = x[1];
      }
    }
    s0 += 64 * ld;
  }
  // operand of MFMA g of tile t; where an edge block's pair was moved back
  // (an odd last row) its first row is the second of the pair
  template <bool EDGE>
  __device__ __forceinline__ double get(int st, int t, int g, bool kin, int lr) const {
    if constexpr (EDGE && T > 1)
      if (!kin && !(t & 1) && 16 * t + 2 * lr == lim - 1) return f[st][t + 1][g];
    return f[st][t][g];
  }
  // the last left < 8 of a product's k: k beyond it read at the chunk's
  // first k and zeroed
  __device__ __forceinline__ void tail(int st, bool kin, bool alt, int lr, int kq, int left) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int k = alt ? 4 * g + kq : 2 * kq + g;
      const bool in = k < left;
      const int ko = in ? 8 * k * (kin ? 1 : ld) : 0;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const double v = ld1(row(t, kin, lr) + ko, s0);
        f[st][t][g] = in ? v : 0.0;
      }
    }
  }
};

// acc += product q, kStages chunks of 8 k, over the first ME x NE tiles of
// the block's MI x NI; CIL: columns interleaved (always where op(B) is
// contiguous in its columns)
template <int MI, int NI, int ME, int NE, bool CIL, bool EDGE>
__device__ __forceinline__ void run_d(v4d* acc, const DProd& q, bool ta, bool tb, int mr, int nr, int m0, int n0) {
  constexpr int S = kStages;
  const int lane = threadIdx.x & 63, lr = lane & 15, kq = lane >> 4;
  const int K = q.k1 - q.k0, n = K >> 3, left = K & 7;
  if (K <= 0) return;
  // MFMA g of a chunk takes k = 4 g + kq where both operands are contiguous
  // in their rows (a last chunk of at most 4 k is one MFMA), else 2 kq + g
  const bool alt = !ta && tb;
  DOperand<ME, S, true> A;
  DOperand<NE, S, CIL> B;
  A.set(q.A, m0, q.k0, q.lda, ta, alt, mr, lr, kq);
  B.set(q.B, n0, q.k0, q.ldb, !tb, alt, nr, lr, kq);
  auto load = [&](int st) {
    A.template load<EDGE>(st, ta, alt, lr, kq);
    B.template load<EDGE>(st, !tb, alt, lr, kq);
  };
  auto mma = [&](int st, int ng) {
#pragma unroll
    for (int g = 0; g < 2; ++g)
      if (g < ng) {
        double a[ME], b[NE];
#pragma unroll
        for (int mi = 0; mi < ME; ++mi) a[mi] = A.template get<EDGE>(st, mi, g, ta, lr);
#pragma unroll
        for (int ni = 0; ni < NE; ++ni) b[ni] = B.template get<EDGE>(st, ni, g, !tb, lr);
#pragma unroll
        for (int mi = 0; mi < ME; ++mi)
#pragma unroll
          for (int ni = 0; ni < NE; ++ni)
            acc[mi * NI + ni] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[ni], a[mi], acc[mi * NI + ni], 0, 0, 0);
      }
  };
#pragma unroll
  for (int st = 0; st < S - 1; ++st)
    if (st < n) load(st);
  int x = 0;
  for (; x + 2 * S - 1 <= n; x += S) {
#pragma unroll
    for (int st = 0; st < S; ++st) {
      load((st + S - 1) % S);
      mma(st, 2);
    }
  }
  // the chunks x .. x + S - 2 are in flight, fewer than S more to load
#pragma unroll
  for (int st = 0; st < 2 * S - 2; ++st) {
    if (x + st + S - 1 < n) load((st + S - 1) % S);
    if (x + st < n) mma(st % S, 2);
  }
  if (left) {
    A.tail(0, ta, alt, lr, kq, left);
    B.tail(0, !tb, alt, lr, kq, left);
    mma(0, alt && left <= 4 ? 1 : 2);
  }
}

// columns of a block are interleaved where an op(B) is contiguous in them
constexpr bool col_interleave(int tt1, int tt2) { return tt1 < 0 || (tt1 & 1) || (tt2 & 1); }

// The block of a matrix of one row or one column (at most 64 elements, one a
// lane; pairs of rows do not exist there): 16 k in flight
__device__ __forceinline__ double dot_d(const DProd& q, int row, int col) {
  constexpr int U = 16;
  const double* a = q.A + (q.ta ? (i64)row * q.lda : row);
  const double* b = q.B + (q.tb ? col : (i64)col * q.ldb);
  const i64 sa = q.ta ? 1 : q.lda, sb = q.tb ? q.ldb : 1;
  double s = 0.0;
  int k = q.k0;
  for (; k + U <= q.k1; k += U) {
    double x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[u] = a[(k + u) * sa];
      y[u] = b[(k + u) * sb];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) s = fma(x[u], y[u], s);
  }
  for (; k < q.k1; ++k) s = fma(a[k * sa], b[k * sb], s);
  return q.scale * s;
}

// acc = product q1 + (nq == 2) q2.scale times q2, q2 first: no load is followed
// by arithmetic on its value.  A block that the edge cuts to at
// most half its rows, or to 16 columns where they are not interleaved, leaves
// the MFMAs of the other half out.
template <int WM, int WN, int TT1, int TT2>
__device__ __forceinline__ void mma_d(v4d* acc, const DProd& q1, const DProd& q2, int nq, int M, int N, int m0,
                                      int n0) {
  constexpr int MI = WM / 16, NI = WN / 16;
  constexpr bool CIL = col_interleave(TT1, TT2);
  const int mr = min(WM, M - m0), nr = min(WN, N - n0);   // rows / columns of the block inside the matrix
  auto run = [&](const DProd& q, bool ta, bool tb) {
    if (mr == WM && nr == WN) run_d<MI, NI, MI, NI, CIL, false>(acc, q, ta, tb, mr, nr, m0, n0);
    else if (CIL || nr > 16) {
      if (MI <= 2 || mr > WM / 2) run_d<MI, NI, MI, NI, CIL, true>(acc, q, ta, tb, mr, nr, m0, n0);
      else if constexpr (MI > 2) run_d<MI, NI, MI / 2, NI, CIL, true>(acc, q, ta, tb, mr, nr, m0, n0);
    } else if constexpr (!CIL) {
      run_d<MI, NI, MI, 1, CIL, true>(acc, q, ta, tb, mr, nr, m0, n0);
    }
  };
  if (nq == 2) {
    run(q2, TT1 < 0 ? q2.ta != 0 : (TT2 >> 1) != 0, TT1 < 0 ? q2.tb != 0 : (TT2 & 1) != 0);
#pragma unroll
    for (int x = 0; x < MI * NI; ++x) acc[x] *= q2.scale;
  }
  run(q1, TT1 < 0 ? q1.ta != 0 : (TT1 >> 1) != 0, TT1 < 0 ? q1.tb != 0 : (TT1 & 1) != 0);
}

// SIG as for k_gemm_t: the transposes of the family's two products as
// constants (bit0 TA1, bit1 TB1, bit2 TA2, bit3 TB2), or SIG < 0: each
// problem's own, read at run time through one body for both products
template <int WM, int WN, int SIG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm_d(
    Slots sl, const GemmProb* probs, const GemmTask* tasks, XcdMap xm, double ascale, double s2scale) {
  constexpr int MI = WM / 16, NI = WN / 16;
  constexpr int T1 = SIG < 0 ? -1 : ((SIG & 1) << 1) | ((SIG >> 1) & 1);
  constexpr int T2 = SIG < 0 ? -1 : (((SIG >> 2) & 1) << 1) | ((SIG >> 3) & 1);
  const int ti = xcd_task(xm, blockIdx.x);
  if (ti < 0) return;
  int inst;
  if (!batch_on(sl.act, inst)) return;
  const GemmTask t = tasks[ti];
  GemmProb pr = probs[t.prob];
  // the byte fields come through vector loads: uniform all the same
  auto uni = [](unsigned char& x) { x = (unsigned char)__builtin_amdgcn_readfirstlane((int)x); };
  uni(pr.ta1); uni(pr.tb1); uni(pr.ta2); uni(pr.tb2);
  uni(pr.sa1); uni(pr.sb1); uni(pr.sa2); uni(pr.sb2);
  uni(pr.sc); uni(pr.mode); uni(pr.upper);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = t.tm * (2 * WM) + (wave >> 1) * WM, n0 = t.tn * (2 * WN) + (wave & 1) * WN;
  if (m0 >= pr.m || n0 >= pr.n) return;   // the waves are independent (no barrier below)
  if (pr.upper && m0 >= n0 + WN) return;  // below the diagonal
  const int kb = pr.kchunk > 0 ? t.ks * pr.kchunk : 0;
  const int ke = pr.kchunk > 0 ? min(pr.k, kb + pr.kchunk) : pr.k;
  v4d acc[MI * NI];
#pragma unroll
  for (int a = 0; a < MI * NI; ++a) acc[a] = v4d{0.0, 0.0, 0.0, 0.0};
  // mode bit3: A is upper triangular (as stored, zero below its diagonal):
  // rows m0.. of op(A) reach only k >= m0 (A as stored) or k < m0 + WM (A
  // transposed)
  const bool tri = pr.mode & 8;
  DProd p1, p2;
  p1.A = slot(sl, pr.sa1, inst) + pr.a1; p1.B = slot(sl, pr.sb1, inst) + pr.b1;
  p1.lda = pr.lda; p1.ldb = pr.ldb; p1.ta = pr.ta1; p1.tb = pr.tb1;
  p1.k0 = (tri && !pr.ta1) ? max(kb, m0) : kb;
  p1.k1 = (tri && pr.ta1) ? min(ke, m0 + WM) : ke;
  p1.scale = 1.0;
  p2.A = slot(sl, pr.sa2, inst) + pr.a2; p2.B = slot(sl, pr.sb2, inst) + pr.b2;
  p2.ta = pr.ta2; p2.tb = pr.tb2;
  if (pr.k2 > 0) {
    // second product with its own K and leading dimensions m, n
    p2.lda = pr.m; p2.ldb = pr.n; p2.k0 = 0; p2.k1 = pr.k2; p2.scale = pr.s2 * ((pr.mode & 64) ? ascale : s2scale);
  } else {
    p2.lda = pr.lda; p2.ldb = pr.ldb;
    p2.k0 = (tri && !pr.ta2) ? max(kb, m0) : kb;
    p2.k1 = (tri && pr.ta2) ? min(ke, m0 + WM) : ke;
    p2.scale = pr.s2 * ((pr.mode == 0 || (pr.mode & 16)) ? s2scale : 1.0);
  }
  double* C = const_cast<double*>(slot(sl, pr.sc, inst)) + pr.c + (i64)t.ks * pr.cstride;
  const double al = pr.mode == 0 ? pr.alpha * ascale
                                  : pr.alpha * ((pr.mode & 1) ? ascale : 1.0) * ((pr.mode & 2) ? s2scale : 1.0);
  const double beta = pr.beta;
  if (pr.m == 1 || pr.n == 1) {
    const int row = m0 + (pr.n == 1 ? lane : 0), col = n0 + (pr.n == 1 ? 0 : lane);
    if (row >= min(pr.m, m0 + WM) || col >= min(pr.n, n0 + WN)) return;
    const double v = al * (dot_d(p1, row, col) + (pr.nprod == 2 ? dot_d(p2, row, col) : 0.0));
    double* c = C + row + (i64)col * pr.ldc;
    *c = beta == 0.0 ? v : v + beta * *c;
    return;
  }
  mma_d<WM, WN, T1, T2>(acc, p1, p2, pr.nprod, pr.m, pr.n, m0, n0);
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ci = (lane >> 4) + 4 * r;
      const int col = n0 + (col_interleave(T1, T2) ? 32 * (ni / 2) + 2 * ci + (ni & 1) : 16 * ni + ci);
      if (col >= pr.n) continue;
#pragma unroll
      for (int mi = 0; mi < MI; mi += 2) {
        const int row = m0 + 16 * mi + 2 * (lane & 15);
        double* c = C + row + (i64)col * pr.ldc;
        v2d v = {al * acc[mi * NI + ni][r], al * acc[(mi + 1) * NI + ni][r]};
        if (row + 1 < pr.m) {
          if (beta != 0.0) v += beta * *reinterpret_cast<v2u*>(c);
          *reinterpret_cast<v2u*>(c) = v;
        } else if (row < pr.m) {
          c[0] = beta == 0.0 ? v[0] : v[0] + beta * c[0];
        }
      }
    }
}

}  // namespace

// tile shapes: 0 64x64, 1 128x64, 2 128x128, 3 64x32, 4 32x64, 5 32x32
// (LDS-staged); 6 128x64, 7 64x64 (register-direct, per wave 64x32 /
// 32x32)
int tile_rows(int tile) { return (tile == 1 || tile == 2 || tile == 6) ? 128 : (tile == 4 || tile == 5 ? 32 : 64); }
int tile_cols(int tile) { return tile == 2 ? 128 : ((tile == 3 || tile == 5) ? 32 : 64); }

template <int TBM, int TBN>
static void launch_sig(int sig, int grid, int ninst, const Slots& sl, const GemmProb* probs, const GemmTask* tasks,
                const XcdMap& xm, hipStream_t s, double ascale, double s2scale) {
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(grid, ninst), dim3(256), 0, s, sl, probs, tasks, xm, ascale, s2scale);
  };
  switch (sig) {
    case 0: go(k_gemm_t<TBM, TBN, 0>); break;
    case 1: go(k_gemm_t<TBM, TBN, 1>); break;
    case 2: go(k_gemm_t<TBM, TBN, 2>); break;
    case 3: go(k_gemm_t<TBM, TBN, 3>); break;
    case 4: go(k_gemm_t<TBM, TBN, 4>); break;
    case 8: go(k_gemm_t<TBM, TBN, 8>); break;
    case 10: go(k_gemm_t<TBM, TBN, 10>); break;
    default: go(k_gemm_t<TBM, TBN, -1>); break;
  }
}

template <int WM, int WN>
static void launch_d(int sig, int grid, int ninst, const Slots& sl, const GemmProb* probs, const GemmTask* tasks,
                     const XcdMap& xm, hipStream_t s, double ascale, double s2scale) {
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, dim3(grid, ninst), dim3(256), 0, s, sl, probs, tasks, xm, ascale, s2scale);
  };
  switch (sig) {
    case 0: go(k_gemm_d<WM, WN, 0>); break;
    case 1: go(k_gemm_d<WM, WN, 1>); break;
    case 2: go(k_gemm_d<WM, WN, 2>); break;
    case 3: go(k_gemm_d<WM, WN, 3>); break;
    case 4: go(k_gemm_d<WM, WN, 4>); break;
    case 8: go(k_gemm_d<WM, WN, 8>); break;
    case 10: go(k_gemm_d<WM, WN, 10>); break;
    default: go(k_gemm_d<WM, WN, -1>); break;
  }
}

// the signatures with specialised kernels
int gemm_sig_supported(int sig) { return (sig >= 0 && sig <= 4) || sig == 8 || sig == 10; }

void launch_gemm_tiled(int tile, const Slots& sl, const GemmProb* probs, const GemmTask* tasks, int grid,
                       const XcdMap& xm, hipStream_t s, double ascale, double s2scale, int ninst, int sig) {
  if (grid <= 0) return;
  if (!gemm_sig_supported(sig)) sig = -1;
  switch (tile) {
    case 0: launch_sig<64, 64>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
    case 1: launch_sig<128, 64>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
    case 3: launch_sig<64, 32>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
    case 4: launch_sig<32, 64>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
    case 5: launch_sig<32, 32>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
    case 6: launch_d<64, 32>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
    case 7: launch_d<32, 32>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
    default: launch_sig<128, 128>(sig, grid, ninst, sl, probs, tasks, xm, s, ascale, s2scale); break;
  }
}

}  // namespace imsrg
