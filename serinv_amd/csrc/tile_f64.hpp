// Single-workgroup FP64 tile factorizations held in LDS (tiles up to 64x64).
//
//   potrf : L = chol(A) (lower, strict upper zero-filled), like
//           scipy.linalg.cholesky(lower=True) which the reference uses
//           (src/serinv/__init__.py:151).  A non-positive or NaN pivot at
//           tile column j records info = row_offset + j + 1 (LAPACK style).
//   trtri : X = L^{-1} for a lower-triangular L (strict upper zero-filled).
//
// Both are blocked by 16 columns.  The sequential part of a 16-column step
// (pivot, scaling, rank-1 updates inside the panel) runs in ONE wave with the
// panel rows spread over the 64 lanes and pivots broadcast by readlane, so it
// needs no workgroup barrier; the trailing updates of the tile are 16x16x4
// FP64 MFMA products spread over the four waves.
#pragma once
#include "common.hpp"

namespace rocbta {

constexpr int TT = 64;  // maximum tile order
constexpr int TT_THREADS = 256;
constexpr int TT_LD = TT + 1;
constexpr int PW = 16;  // panel width

struct TileBatch {
  double* A;         // tile (0,0) of batch entry 0
  int64_t lda;
  int64_t sA1, sA2;  // batch strides
  double* X;         // optional output (inverse); may alias nothing in A
  int64_t ldx;
  int64_t sX1, sX2;
  int m;             // tile order (<= 64)
  int batch1, batch2;
  int* info;
  int64_t info_row0;       // global row of the tile's first row, for info
  int64_t info_s1, info_s2;  // global-row strides along the batch dims
  // Strict-upper zero fill of the rows of the tile that lie right of it:
  // zcols columns starting at column m of each tile row (0 = none).
  int zcols;
  int mode;         // list launches: 0 potrf (+ inverse), 1 inverse only
  int grid_begin;   // list launches: first workgroup of this entry
};

// Wave of the calling lane as a scalar: branches on it are scalar branches, and
// what one wave keeps in registers does not count in another wave's branch.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// Lane index as a new value at each call: addresses formed from it are computed
// where they are used.  In a long loop the compiler otherwise forms all of
// them once before it and runs out of registers.
__device__ __forceinline__ int fresh_lane() {
  int l = threadIdx.x & 63;
  asm volatile("" : "+v"(l));
  return l;
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// d = sqrt(x), inv = 1/sqrt(x) for x > 0 (NaN propagates), from the hardware
// reciprocal square root y0 (relative error below 2^-22) and one third-order
// correction of it: with e = 1 - x y0^2,
//   1/sqrt(x) = y0 (1 - e)^(-1/2) = y0 (1 + e/2 + 3e^2/8 + O(e^3)),
// so y = y0 + (y0 e)(1/2 + 3e/8) leaves a relative error of about 2.5 * 2^-66
// before rounding (four dependent operations after the seed; two Newton
// steps take six).  The square root is one Newton step on d = x y,
// d <- d + y (x - d^2) / 2, which is not on the path of inv.
__device__ __forceinline__ void pivot_sqrt(double x, double& d, double& inv) {
  const double y0 = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y0), y0, 1.0);
  const double p = __builtin_fma(0.375, e, 0.5);
  const double y = __builtin_fma(y0 * e, p, y0);
  double s = x * y;
  const double rr = __builtin_fma(-s, s, x);
  s = __builtin_fma(0.5 * y, rr, s);
  d = s;
  inv = y;
}

// Unblocked Cholesky of the panel S[p:m, p:p+w] (w <= 16, m - p <= 64) by
// the calling wave; lane l owns row p + l.  Lower entries are written back.
template <int WFIX>
__device__ __forceinline__ void wave_panel_potrf(double (*S)[TT_LD], int p, int m, int w_rt,
                                                 int* info, int64_t row0) {
  const int w = WFIX ? WFIX : w_rt;
  const int lane = threadIdx.x & 63;
  const int i = p + lane;
  const bool act = i < m;
  double r[PW];
#pragma unroll
  for (int k = 0; k < PW; ++k) r[k] = (act && k < w) ? S[i][p + k] : 0.0;
#pragma unroll
  for (int j = 0; j < PW; ++j) {
    if (j < w) {
      double piv = readlane_f64(r[j], j);
      if (!(piv > 0.0)) {
        if (lane == 0) record_info(info, (int)(row0 + p + j + 1));
        piv = __builtin_nan("");
      }
      double d, inv;
      pivot_sqrt(piv, d, inv);
      // the column is broadcast from its scaled value; the diagonal entry d
      // (lane j) is not on the path to the next pivot
      const double sc = r[j] * inv;
#pragma unroll
      for (int k = j + 1; k < PW; ++k) {
        if (k < w) {
          const double lkj = readlane_f64(sc, k);
          r[k] -= sc * lkj;
        }
      }
      r[j] = (lane == j) ? d : (lane > j ? sc : r[j]);
    }
  }
#pragma unroll
  for (int k = 0; k < PW; ++k)
    if (act && k < w && p + k <= i) S[i][p + k] = r[k];
}

// Value of lane K of each 16-lane row, in every lane of the row.  The wait
// states in front of a DPP read are written out (here and in row_fmac): the
// compiler does not track that hazard into an asm statement.
template <int K>
__device__ __forceinline__ double row_bcast(double v) {
  double r;
  asm volatile("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
               : "=v"(r)
               : "v"(v), "n"(K));
  return r;
}
// Lane K of a and of b.
template <int K>
__device__ __forceinline__ void row_bcast2(double a, double b, double& ra, double& rb) {
  asm volatile(
      "s_nop 1\n\tv_mov_b64_dpp %0, %2 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b64_dpp %1, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf"
      : "=&v"(ra), "=v"(rb)
      : "v"(a), "v"(b), "n"(K));
}

// x[K0 + i] -= s[lane K0 + i of the row] * y for i < N: one v_fmac_f64_dpp
// each, the row broadcast being an operand modifier.  Eight share one wait,
// which costs as much as two of them.
#define ROCBTA_FMAC(x, k) \
  "v_fmac_f64_dpp " x ", -%[s], %[y] row_newbcast:%[k]+" k " row_mask:0xf bank_mask:0xf\n\t"
#define ROCBTA_IN : [s] "v"(s), [y] "v"(y), [k] "n"(K0)
template <int K0, int N>
__device__ __forceinline__ void row_fmac(double (&x)[PW], double s, double y) {
  if constexpr (N == 1) {
    asm volatile("s_nop 1\n\t" ROCBTA_FMAC("%0", "0") : "+v"(x[K0]) ROCBTA_IN);
  } else if constexpr (N == 2) {
    asm volatile("s_nop 1\n\t" ROCBTA_FMAC("%0", "0") ROCBTA_FMAC("%1", "1")
                 : "+v"(x[K0]), "+v"(x[K0 + 1]) ROCBTA_IN);
  } else if constexpr (N == 3) {
    asm volatile("s_nop 1\n\t" ROCBTA_FMAC("%0", "0") ROCBTA_FMAC("%1", "1") ROCBTA_FMAC("%2", "2")
                 : "+v"(x[K0]), "+v"(x[K0 + 1]), "+v"(x[K0 + 2]) ROCBTA_IN);
  } else if constexpr (N >= 4 && N < 8) {
    asm volatile("s_nop 1\n\t" ROCBTA_FMAC("%0", "0") ROCBTA_FMAC("%1", "1") ROCBTA_FMAC("%2", "2")
                     ROCBTA_FMAC("%3", "3")
                 : "+v"(x[K0]), "+v"(x[K0 + 1]), "+v"(x[K0 + 2]), "+v"(x[K0 + 3]) ROCBTA_IN);
    row_fmac<K0 + 4, N - 4>(x, s, y);
  } else if constexpr (N >= 8) {
    asm volatile("s_nop 1\n\t" ROCBTA_FMAC("%0", "0") ROCBTA_FMAC("%1", "1") ROCBTA_FMAC("%2", "2")
                     ROCBTA_FMAC("%3", "3") ROCBTA_FMAC("%4", "4") ROCBTA_FMAC("%5", "5")
                         ROCBTA_FMAC("%6", "6") ROCBTA_FMAC("%7", "7")
                 : "+v"(x[K0]), "+v"(x[K0 + 1]), "+v"(x[K0 + 2]), "+v"(x[K0 + 3]),
                   "+v"(x[K0 + 4]), "+v"(x[K0 + 5]), "+v"(x[K0 + 6]), "+v"(x[K0 + 7]) ROCBTA_IN);
    row_fmac<K0 + 8, N - 8>(x, s, y);
  }
}
#undef ROCBTA_IN
#undef ROCBTA_FMAC

// Column J of the panel: x is its pivot (in every lane).  The steps of the
// reciprocal square root (pivot_sqrt) are a dependent chain; the updates by
// column J - 1, still open when column J starts, are dealt between them in
// this order (the scheduling barriers keep it).  The next pivot is formed from
// two broadcasts, A(J+1,J) and A(J+1,J+1), read ahead of the root, so neither
// the scaled column nor a broadcast of it is on the path from pivot to pivot.
// pv: lane J keeps its pivot.
template <int J>
__device__ __forceinline__ void panel_columns(double (&d)[PW], double (&r)[PW], double x,
                                              double& pv, bool ident, int li) {
  if constexpr (J < PW) {
    constexpr int N = J == 0 ? 0 : PW - J;  // open updates of d[J ..] and of r[J ..]
    constexpr int N1 = N < 8 ? N / 2 : N - 8;
    constexpr int JP = J == 0 ? 0 : J - 1, JN = J + 1 < PW ? J + 1 : J;
    const double sp = d[JP], srp = r[JP];
    double u = 0.0, nx = 0.0;
    __builtin_amdgcn_sched_barrier(0);
    const double y0 = __builtin_amdgcn_rsq(x);
    __builtin_amdgcn_sched_barrier(0);
    row_fmac<J, N>(d, sp, sp);
    __builtin_amdgcn_sched_barrier(0);
    const double t = x * y0;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (J + 1 < PW) row_bcast2<JN>(d[J], d[JN], u, nx);
    __builtin_amdgcn_sched_barrier(0);
    const double e = __builtin_fma(-t, y0, 1.0);
    __builtin_amdgcn_sched_barrier(0);
    row_fmac<J, N1>(r, sp, srp);
    if constexpr (J == 0) {
      // the rows of the identity (see wave_panel_potrf16)
#pragma unroll
      for (int k = 0; k < PW; ++k) r[k] = ident ? (k == li ? 1.0 : 0.0) : r[k];
    }
    __builtin_amdgcn_sched_barrier(0);
    const double q = y0 * e;
    const double p = __builtin_fma(0.375, e, 0.5);
    __builtin_amdgcn_sched_barrier(0);
    row_fmac<J + N1, N - N1>(r, sp, srp);
    __builtin_amdgcn_sched_barrier(0);
    const double y = __builtin_fma(q, p, y0);
    pv = li == J ? x : pv;
    __builtin_amdgcn_sched_barrier(0);
    const double w = u * y;
    d[J] *= y;
    __builtin_amdgcn_sched_barrier(0);
    const double xn = __builtin_fma(-w, w, nx);
    r[J] *= y;
    __builtin_amdgcn_sched_barrier(0);
    panel_columns<J + 1>(d, r, xn, pv, ident, li);
  }
}

// Cholesky of the 16-column panel S[p:m, p:p+16] (p + 16 <= m <= 64) by one
// wave, and, with INV, the inverse of its diagonal block (16 x 16, zeros above
// the diagonal).  factor() leaves the rows below the diagonal block in S;
// finish() writes the block, and its inverse to Xp (row pitch ldx), which may
// wait until other waves have been let on to those rows.
//
// Every 16-lane row of the wave holds the diagonal block (lane li of the row:
// matrix row p + li, in d), so the broadcast of a column entry is the
// row_newbcast modifier of a multiply-add and costs no instruction.  Beside
// it, r holds one further row per lane that is solved against the block as it
// is factored: lanes 16 .. 63 the panel rows below it, lanes 0 .. 15 the
// identity, whose solution is the transposed inverse of the block.
//
// Bound by FP64 issue on one wave: 272 multiply-adds of 4 cycles and 16
// dependent pivot steps of about 80.  Entries of S above the diagonal of the
// block are left undefined.  A non-positive or NaN pivot turns into NaN
// through the reciprocal square root, so the loop has no branch; the first
// failing column is recorded once after it.
template <bool INV>
struct WavePanel16 {
  double d[PW], r[PW], pv;
  __device__ __forceinline__ void factor(double (*S)[TT_LD], int p, int m) {
    const int lane = fresh_lane(), li = lane & 15;
    const int row = p + lane;
    const double* sd = &S[p + li][p];
    const double* sr = &S[row < m ? row : p + li][p];
#pragma unroll
    for (int k = 0; k < PW; ++k) d[k] = sd[k];
#pragma unroll
    for (int k = 0; k < PW; ++k) r[k] = sr[k];
    pv = 0.0;
    panel_columns<0>(d, r, row_bcast<0>(d[0]), pv, INV && lane < 16, li);
    if (lane >= 16 && row < m) {
      double* dst = &S[row][p];
#pragma unroll
      for (int k = 0; k < PW; ++k) dst[k] = r[k];
    }
  }
  __device__ __forceinline__ void finish(double (*S)[TT_LD], int p, double* Xp, int ldx, int* info,
                                         int64_t row0) {
    const int lane = fresh_lane();
    if (lane < 16) {
      if (INV) {
#pragma unroll
        for (int k = 0; k < PW; ++k) Xp[k * ldx + lane] = r[k];
      }
      double* dst = &S[p + lane][p];
#pragma unroll
      for (int k = 0; k < PW; ++k) dst[k] = d[k];
      double s, inv;
      pivot_sqrt(pv, s, inv);
      dst[lane] = s;
    }
    const uint64_t bad = __ballot(!(pv > 0.0)) & 0xffffull;
    if (bad && lane == 0) record_info(info, (int)(row0 + p + __builtin_ctzll(bad) + 1));
  }
};

// S[q:m, q:m] (lower part) -= P P^T with P = S[q:m, p:p+w], on MFMA, all
// waves.  Output 16x16 blocks are dealt round-robin to the waves.
template <int WFIX>
__device__ __forceinline__ void lds_syrk_update(double (*S)[TT_LD], int p, int w_rt, int q,
                                                int m) {
  const int w = WFIX ? WFIX : w_rt;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nb = (m - q + 15) / 16;
  const int li = lane & 15, lk = lane >> 4;
  int t = 0;
  for (int bi = 0; bi < nb; ++bi)
    for (int bj = 0; bj <= bi; ++bj, ++t) {
      if ((t & 3) != wave) continue;
      f64x4 acc = {0.0, 0.0, 0.0, 0.0};
      const int ra = q + bi * 16 + li, rb = q + bj * 16 + li;
#pragma unroll
      for (int kk = 0; kk < PW; kk += 4) {
        const int k = kk + lk;
        const double av = (k < w && ra < m) ? S[ra][p + k] : 0.0;
        const double bv = (k < w && rb < m) ? S[rb][p + k] : 0.0;
        acc = mfma_f64(av, bv, acc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = q + bi * 16 + acc_row_f64(lane, r);
        const int col = q + bj * 16 + acc_col(lane);
        if (row < m && col <= row) S[row][col] -= acc[r];
      }
    }
}

// Full 64-tile form: S[c0:64, c0:c1] (lower 16 x 16 blocks) -= P P^T
// restricted to the 16-wide column blocks [c0, c1), P = S[:, p:p+16].  Block t
// of the enumeration goes to wave wave0 + t % nw; other waves return at once.
// Diagonal blocks are written in full (nothing reads a tile above its
// diagonal).
__device__ __forceinline__ void lds_syrk_cols(double (*S)[TT_LD], int p, int c0, int c1,
                                              int wave0, int nw) {
  const int lane = fresh_lane(), wave = wave_id();
  const int li = lane & 15, lk = lane >> 4;
  int t = 0;
  for (int cb = c0 / 16; cb < c1 / 16; ++cb)
    for (int rb = cb; rb < TT / 16; ++rb, ++t) {
      if (wave != wave0 + t % nw) continue;
      const double* ra = &S[rb * 16 + li][p + lk];
      const double* rc = &S[cb * 16 + li][p + lk];
      double av[4], bv[4], cv[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        av[k] = ra[4 * k];
        bv[k] = rc[4 * k];
      }
      double* c = &S[rb * 16 + lk][cb * 16 + li];  // accumulator register r: row + 4 r
#pragma unroll
      for (int r = 0; r < 4; ++r) cv[r] = c[4 * r * TT_LD];
      f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 4; ++k) acc = mfma_f64(av[k], bv[k], acc);
#pragma unroll
      for (int r = 0; r < 4; ++r) c[4 * r * TT_LD] = cv[r] - acc[r];
    }
}

struct NoIdle {
  __device__ void operator()(int) const {}
};

// Blocked Cholesky of S (m x m, lower part valid) in place.  MFIX = 64
// compiles the full-tile case with all sizes constant and a look-ahead: after
// panel p only the next panel's columns are updated (waves 1-3) before the
// next panel is factored (wave 0), while waves 1-3 apply panel p to the
// columns beyond it.  Full tiles also leave the inverses of the four diagonal
// blocks in X's (each written with its panel), and after the update beside a
// panel, waves 1-3 run idle(p) while wave 0 factors panel p + 16, from p = -16
// on; panels 0 .. p and their blocks' inverses are final by then.  Columns 16
// .. 63 of S may be completed by idle(-16).  The call ends with a barrier
// after the last of them.  MFIX = 0 handles any m <= 64 and leaves X alone.
template <int MFIX, typename IDLE = NoIdle>
__device__ __forceinline__ void lds_potrf_t(double (*S)[TT_LD], double (*X)[TT_LD], int m_rt,
                                            int* info, int64_t row0, IDLE idle = IDLE()) {
  const int m = MFIX ? MFIX : m_rt;
  const int wave = wave_id();
  if (MFIX == TT) {
    WavePanel16<true> w;
    if (wave == 0)
      w.factor(S, 0, TT);
    else
      idle(-PW);
    __syncthreads();
#pragma unroll
    for (int p = 0; p + PW < TT; p += PW) {
      if (wave == 0)
        w.finish(S, p, &X[p][p], TT_LD, info, row0);
      else
        lds_syrk_cols(S, p, p + PW, p + 2 * PW, 1, 3);  // next panel's columns
      __syncthreads();
      if (wave == 0) {
        w.factor(S, p + PW, TT);
        if (p + 2 * PW == TT) w.finish(S, p + PW, &X[p + PW][p + PW], TT_LD, info, row0);
      } else {
        if (p + 2 * PW < TT) lds_syrk_cols(S, p, p + 2 * PW, TT, 1, 3);  // the rest, beside the panel
        idle(p);
      }
      __syncthreads();
    }
    return;
  }
#pragma unroll
  for (int p = 0; p < m; p += PW) {
    const int w = min(PW, m - p);
    if (w == PW) {
      if (wave == 0) {
        WavePanel16<false> wp;
        wp.factor(S, p, m);
        wp.finish(S, p, nullptr, 0, info, row0);
      }
    } else {
      if (wave == 0) wave_panel_potrf<0>(S, p, m, w, info, row0);
    }
    __syncthreads();
    if (p + w < m) {
      lds_syrk_update<0>(S, p, w, p + w, m);
      __syncthreads();
    }
  }
}

__device__ __forceinline__ void lds_potrf(double (*S)[TT_LD], double (*X)[TT_LD], int m, int* info,
                                          int64_t row0) {
  if (m == TT)
    lds_potrf_t<TT>(S, X, TT, info, row0);
  else
    lds_potrf_t<0>(S, X, m, info, row0);
}

// X = L^{-1} (m x m lower, in S) into Xs (lower; strict upper zero).
// Step 1: each wave inverts 16x16 diagonal blocks (full tiles: as the rows
// of a triangular solve; ragged ones by Gauss-Jordan sweeps, lane = (row i,
// column group g of four columns)).  Step 2: off-diagonal blocks by
// increasing distance d from the diagonal on MFMA:
//   X_IJ = -X_II * sum_{K=J}^{I-1} L_IK X_KJ.
// Ws: 64 x 17 scratch of the ragged form; at distance d the block (I, I-d) of
// W sits in rows 16I .. 16I+15.
constexpr int WS_LD = 17;

// Columns J .. 15 of r <- r L^{-T} for the 16 x 16 lower triangle whose rows
// lie in d (replicated in every 16-lane row) and whose inverse diagonal lies
// in dinv, lane = row.
template <int J>
__device__ __forceinline__ void trinv_columns(const double (&d)[PW], double (&r)[PW], double dinv) {
  if constexpr (J < PW) {
    r[J] *= row_bcast<J>(dinv);
    row_fmac<(J + 1 < PW ? J + 1 : J), PW - 1 - J>(r, d[J], r[J]);
    trinv_columns<J + 1>(d, r, dinv);
  }
}

// Inverse of the full 16x16 lower-triangular block of S at (o, o) by the
// calling wave, written to dst (row pitch ld) as a full block (zeros above
// the diagonal): the rows of the identity solved against the block give the
// rows of its transposed inverse, with the broadcasts of a column as operand
// modifiers (row_fmac), 120 multiply-adds in all.  Lanes 16 .. 63 repeat
// lanes 0 .. 15.  Measured with the block in LDS: 2939 cycles before (column
// substitution on LDS broadcasts).
__device__ __forceinline__ void wave_diag_inv16_to(const double (*S)[TT_LD], int o, double* dst,
                                                   int ld) {
  const int lane = threadIdx.x & 63, li = lane & 15;
  double d[PW], r[PW];
  const double dinv = 1.0 / S[o + li][o + li];
#pragma unroll
  for (int k = 0; k < PW; ++k) d[k] = S[o + li][o + k];
#pragma unroll
  for (int k = 0; k < PW; ++k) r[k] = k == li ? 1.0 : 0.0;
  trinv_columns<0>(d, r, dinv);
  if (lane < 16) {
#pragma unroll
    for (int k = 0; k < PW; ++k) dst[k * ld + li] = r[k];
  }
}
__device__ __forceinline__ void wave_diag_inv16(const double (*S)[TT_LD], double (*Xs)[TT_LD],
                                                int o) {
  wave_diag_inv16_to(S, o, &Xs[o][o], TT_LD);
}

// Off-diagonal 16x16 block of X = L^{-1} by the calling wave (J < I):
//   X_IJ = -X_II * W,  W = sum_{K=J}^{I-1} L_IK X_KJ,
// with L in S, the blocks X_KJ (K < I) in Xs, and X_II read from XI (row
// pitch ldi).  X_IJ is written to Xs.  Lane (q, j) = (lane >> 4, lane & 15)
// holds W(4r + q, j) in w[r] after the first product, which is the B operand
// of k-step r of the second, so W never leaves the registers.
__device__ __forceinline__ void wave_trtri_offdiag(const double (*S)[TT_LD], double (*Xs)[TT_LD],
                                                   const double* XI, int ldi, int I, int J) {
  const int lane = fresh_lane(), li = lane & 15, lk = lane >> 4;
  f64x4 w = {0.0, 0.0, 0.0, 0.0};
  for (int K = J; K < I; ++K)
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4) {
      const int k = K * 16 + kk + lk;
      w = mfma_f64(S[I * 16 + li][k], Xs[k][J * 16 + li], w);
    }
  f64x4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < 4; ++r) x = mfma_f64(XI[li * ldi + 4 * r + lk], w[r], x);
#pragma unroll
  for (int r = 0; r < 4; ++r) Xs[I * 16 + acc_row_f64(lane, r)][J * 16 + acc_col(lane)] = -x[r];
}

// Blocks 0 .. I - 1 of block row I of X = L^{-1} by the calling wave, as
// wave_trtri_offdiag with X_II in Xs, in two parts: the products W_J = sum_K
// L_IK X_KJ need block row I of L up to column I - 1 only, so they can run
// while block (I, I) is factored.  All operands are read before the first MFMA
// and the chains of dependent MFMAs run interleaved.
template <int I>
struct WaveTrtriRow {
  f64x4 w[I];
  __device__ __forceinline__ void products(const double (*S)[TT_LD], const double (*Xs)[TT_LD]) {
    const int lane = fresh_lane(), li = lane & 15, lk = lane >> 4;
    double a[I][4], b[I][I][4];
#pragma unroll
    for (int k = 0; k < I; ++k)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[k][u] = S[I * 16 + li][k * 16 + 4 * u + lk];
#pragma unroll
        for (int j = 0; j <= k; ++j) b[j][k][u] = Xs[k * 16 + 4 * u + lk][j * 16 + li];
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < I; ++j) w[j] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < I; ++k)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int j = 0; j <= k; ++j) w[j] = mfma_f64(a[k][u], b[j][k][u], w[j]);
  }
  __device__ __forceinline__ void finish(double (*Xs)[TT_LD]) const {
    const int lane = fresh_lane(), li = lane & 15, lk = lane >> 4;
    double xi[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) xi[r] = Xs[16 * I + li][16 * I + 4 * r + lk];
    f64x4 x[I];
#pragma unroll
    for (int j = 0; j < I; ++j) x[j] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < I; ++j) x[j] = mfma_f64(xi[r], w[j][r], x[j]);
#pragma unroll
    for (int j = 0; j < I; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        Xs[I * 16 + acc_row_f64(lane, r)][j * 16 + acc_col(lane)] = -x[j][r];
  }
};

// ZERO = false: the caller guarantees that the blocks of Xs strictly above
// the 16x16 block diagonal already hold zeros (they are never written here).
// DIAG = false (full tiles): the inverses of the diagonal blocks are there.
template <int MFIX, bool ZERO = true, bool DIAG = true>
__device__ __forceinline__ void lds_trtri_t(const double (*S)[TT_LD], double (*Xs)[TT_LD],
                                            double (*Ws)[WS_LD], int m_rt) {
  const int m = MFIX ? MFIX : m_rt;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tid = threadIdx.x;
  if (ZERO || !MFIX) {
    for (int idx = tid; idx < TT * TT; idx += TT_THREADS) Xs[idx / TT][idx % TT] = 0.0;
    __syncthreads();
  }
  if (MFIX == TT) {
    if (DIAG) {
      wave_diag_inv16(S, Xs, __builtin_amdgcn_readfirstlane(16 * wave));
      __syncthreads();
    }
#pragma unroll
    for (int dist = 1; dist < TT / 16; ++dist) {
      const int I = wave + dist;
      if (I < TT / 16) wave_trtri_offdiag(S, Xs, &Xs[16 * I][16 * I], TT_LD, I, wave);
      __syncthreads();
    }
    return;
  }
  const int nb = (m + 15) / 16;
  for (int blk = wave; blk < nb; blk += 4) {
    const int o = blk * 16, w = min(16, m - o);
    const int i = lane & 15, g = lane >> 4;
    double x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = (i == g * 4 + q) ? 1.0 : 0.0;
    for (int j = 0; j < w; ++j) {
      if (i == j) {
        const double inv = 1.0 / S[o + j][o + j];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] *= inv;
      }
      const double lij = (i > j && i < w) ? S[o + i][o + j] : 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double xj = __shfl(x[q], g * 16 + j, 64);
        x[q] -= lij * xj;
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = g * 4 + q;
      if (i < w && c < w && c <= i) Xs[o + i][o + c] = x[q];
    }
  }
  __syncthreads();
  const int li = lane & 15, lk = lane >> 4;
  for (int d = 1; d < nb; ++d) {
    // W_J = sum_{K=J}^{J+d-1} L_{J+d,K} X_{K,J}  (into Ws block row J+d, col J)
    for (int J = wave; J + d < nb; J += 4) {
      const int I = J + d;
      f64x4 acc = {0.0, 0.0, 0.0, 0.0};
      for (int K = J; K < I; ++K)
#pragma unroll
        for (int kk = 0; kk < 16; kk += 4) {
          const int k = K * 16 + kk + lk;
          const int ra = I * 16 + li, cb = J * 16 + li;
          const double av = (ra < m && k < m) ? S[ra][k] : 0.0;
          const double bv = (k < m && cb < m) ? Xs[k][cb] : 0.0;
          acc = mfma_f64(av, bv, acc);
        }
#pragma unroll
      for (int r = 0; r < 4; ++r) Ws[I * 16 + acc_row_f64(lane, r)][acc_col(lane)] = acc[r];
    }
    __syncthreads();
    for (int J = wave; J + d < nb; J += 4) {
      const int I = J + d;
      f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int kk = 0; kk < 16; kk += 4) {
        const int k = I * 16 + kk + lk;
        const int ra = I * 16 + li;
        const double av = (ra < m && k < m) ? Xs[ra][k] : 0.0;
        const double bv = (k < m) ? Ws[k][li] : 0.0;
        acc = mfma_f64(av, bv, acc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = I * 16 + acc_row_f64(lane, r), col = J * 16 + acc_col(lane);
        if (row < m && col < m) Xs[row][col] = -acc[r];
      }
    }
    __syncthreads();
  }
}

template <bool ZERO = true>
__device__ __forceinline__ void lds_trtri(const double (*S)[TT_LD], double (*Xs)[TT_LD],
                                          double (*Ws)[WS_LD], int m) {
  if (m == TT)
    lds_trtri_t<TT, ZERO>(S, Xs, Ws, TT);
  else
    lds_trtri_t<0>(S, Xs, Ws, m);
}

// mode 0: potrf (+ inverse into X if X != nullptr); mode 1: trtri only.
template <int MODE>
__device__ __forceinline__ void tile_factor_body(const TileBatch& tb, int bz, double (*S)[TT_LD],
                                                 double (*Xs)[TT_LD], double (*Ws)[WS_LD]) {
  const int b1 = bz % tb.batch1, b2 = bz / tb.batch1;
  double* A = tb.A + b1 * tb.sA1 + b2 * tb.sA2;
  const int m = tb.m;
  const int tid = threadIdx.x;
  for (int idx = tid; idx < TT * TT; idx += TT_THREADS) {
    int r = idx / TT, c = idx % TT;
    double v = 0.0;
    if (r < m && c <= r) v = A[(int64_t)r * tb.lda + c];
    S[r][c] = v;
  }
  if (MODE == 0 && m == TT) {  // the factorization fills in the diagonal blocks' inverses
    for (int idx = tid; idx < TT * TT; idx += TT_THREADS) Xs[idx / TT][idx % TT] = 0.0;
  }
  __syncthreads();
  if (MODE == 0) {
    lds_potrf(S, Xs, m, tb.info, tb.info_row0 + b1 * tb.info_s1 + b2 * tb.info_s2);
    // write L back, upper triangle zero-filled
    for (int idx = tid; idx < m * m; idx += TT_THREADS) {
      int r = idx / m, c = idx % m;
      A[(int64_t)r * tb.lda + c] = (c <= r) ? S[r][c] : 0.0;
    }
    if (tb.zcols > 0) {
      for (int r = 0; r < m; ++r)
        for (int c = tid; c < tb.zcols; c += TT_THREADS) A[(int64_t)r * tb.lda + m + c] = 0.0;
    }
  }
  if (tb.X != nullptr) {
    if (MODE == 0 && m == TT)
      lds_trtri_t<TT, false, false>(S, Xs, Ws, TT);
    else
      lds_trtri(S, Xs, Ws, m);
    double* X = tb.X + b1 * tb.sX1 + b2 * tb.sX2;
    for (int idx = tid; idx < m * m; idx += TT_THREADS) {
      int r = idx / m, c = idx % m;
      X[(int64_t)r * tb.ldx + c] = Xs[r][c];
    }
  }
}

template <int MODE>
__global__ void __launch_bounds__(TT_THREADS) tile_factor_kernel(TileBatch tb) {
  __shared__ double S[TT][TT_LD];
  __shared__ double Xs[TT][TT_LD];
  __shared__ double Ws[TT][WS_LD];
  tile_factor_body<MODE>(tb, blockIdx.x, S, Xs, Ws);
}

// The same over a device array of entries sorted by grid_begin (batched
// plans); each entry runs in its own mode.
__global__ void __launch_bounds__(TT_THREADS) tile_factor_list_kernel(const TileBatch* tbs,
                                                                      int ntb) {
  __shared__ double S[TT][TT_LD];
  __shared__ double Xs[TT][TT_LD];
  __shared__ double Ws[TT][WS_LD];
  const int wg = blockIdx.x;
  int lo = 0, hi = ntb - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tbs[mid].grid_begin <= wg) lo = mid; else hi = mid - 1;
  }
  const TileBatch& tb = tbs[lo];
  if (tb.mode == 0)
    tile_factor_body<0>(tb, wg - tb.grid_begin, S, Xs, Ws);
  else
    tile_factor_body<1>(tb, wg - tb.grid_begin, S, Xs, Ws);
}

}  // namespace rocbta
