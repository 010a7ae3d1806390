// Grouped, batched FP64 MFMA GEMM for gfx950.
//
//   C[p] = beta_p * C[p] + sum_t alpha_t * op(A_t) * op(B_t)      (up to 2 terms)
//
// One launch runs up to ROCBTA_MAX_PROBLEMS independent problems (each with a
// 2-D batch); every workgroup of 8 waves owns one square tile of one C.
// Operands are row-major with leading dimensions; op() is the identity or the
// transpose.  Triangular operands (a stored triangle of zeros) shorten the K
// loop.  `uplo` restricts the written part of C to its lower (or upper)
// triangle, which is how the symmetric rank-k (syrk-type) updates are expressed.
//
// Aliasing contract: C may alias an operand of a term only when the problem
// is a single 64-wide tile across (N <= 64 for A, M <= 64 for B) and the launch
// uses 64-wide tiles: a workgroup then owns all of C that it reads, and reads
// all of it before it writes.
//
// Every wave computes a 32 x 32 block of the tile over its share of the K
// range, with the MFMA operands loaded straight from global memory: an FP64
// MFMA step takes 64 cycles on its SIMD, so a wave needs 4 KiB of operands per
// 512 cycles, which the caches deliver without staging them in LDS, and the
// waves run without a barrier until their blocks are summed.  Bound by the
// MFMA pipes for large products (63 TFLOP/s is 88% of what they reach at the
// clock held), by the L1's load path behind them and, for small ones, by the
// round trips of a launch: two groups in flight at four waves per SIMD measured
// best (three or four groups at two waves per SIMD: 640 against 581 us for
// sixteen 1024^3 products).  Measured, against the LDS-staged 64-tile kernel before
// (A and B as they are / B transposed / A transposed): 64^3 4.6 / 4.8 / 4.5
// (9.5) us, 512^3 10.2 / 10.6 / 10.0 (26.5) us, 1024^3 46 / 49 / 44 (52 / 50 /
// 51) us, sixteen 1024^3 551 / 578 / 544 (630 / 626 / 628) us; FP32 products,
// sixteen 1024^3 429 / 486 / 402 (457 / 444 / 436) us.
#pragma once
#include "common.hpp"

namespace rocbta {

constexpr int GT_THREADS = 512;  // 8 waves
constexpr int GT_WAVES = GT_THREADS / 64;
constexpr int GW = 32;   // rows and columns of a wave's block
constexpr int GK = 16;   // k indices per load group
constexpr int GPF = 2;   // load groups in flight per wave
constexpr int GP = GW + 2;  // LDS pitch of a block (doubles)
#define ROCBTA_MAX_PROBLEMS 4

enum Tri : uint8_t { TRI_NONE = 0, TRI_LOWER = 1, TRI_UPPER = 2 };

struct GemmTerm {
  const double* A;
  const double* B;
  int64_t lda, ldb;
  int64_t sA1, sA2, sB1, sB2;  // batch strides (elements) along batch dims 1 and 2
  double alpha;
  // (whole words: scalar loads read no bytes)
  int K;
  int transA, transB;
  int triA;  // shape of op(A): TRI_LOWER => op(A)(m,k) = 0 for k > m
  int triB;  // shape of op(B): TRI_LOWER => op(B)(k,n) = 0 for k < n
};

struct GemmProblem {
  double* C;
  int64_t ldc;
  int64_t sC1, sC2;
  int M, N;
  int batch1, batch2;
  double beta;
  int nterms;
  int uplo;    // TRI_NONE: full C; TRI_LOWER: only row >= col is written
  int mirror;  // with uplo == TRI_LOWER: also write C[col][row] = C[row][col]
  int tiles_m, tiles_n;
  // lower_packed (uplo == TRI_LOWER, tiles_m == tiles_n): a batch entry has
  // tiles_m (tiles_m + 1) / 2 workgroups, one per lower tile, instead of
  // tiles_m * tiles_n of which the upper ones would exit at once.
  int lower_packed;
  int tile_begin;  // first global tile index of this problem
  // Mixed precision: operands are read as FP64 and rounded to FP32 at the
  // MFMA, products accumulate in FP32 (v_mfma_f32_16x16x4_f32); the sum over
  // the waves and the epilogue (beta * C + result) run in FP64.
  int f32;
  GemmTerm t[2];
};

struct GemmGroup {
  int nprob;
  int total_tiles;
  GemmProblem p[ROCBTA_MAX_PROBLEMS];
};

typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef double dbl2u __attribute__((ext_vector_type(2), aligned(8)));  // any double address

// --------------------------------------------------------------- operands
// Operand element (r, k), r in the wave's 32 rows (columns, for B), is stored
// at p[r * ld + k] (KC: contiguous in k) or p[k * ld + r].  Lane (li, lk) of
// sub-block i holds r = 2 li + i, and on MFMA step s of a group of 16 k
//   k = k0 + 8 (s >> 1) + 2 lk + (s & 1),
// the same for both operands (which of the four k of a step sits in which
// lane group is free).  Either storage then takes four 16-byte loads per lane
// and group: one per k (256 contiguous bytes per k), or, KC, one per row of four
// (128 contiguous bytes of eight rows), two adjacent lanes on one line, which then
// trade (frag_trade).  What a load costs is the lines among neighbouring lanes:
// with a row per lane, 64 bytes of sixteen rows a load, sixteen 1024^3 products
// took 598 us with one operand stored this way and 892 us with both (551 and 578
// so); with lanes four apart on one line it was 593 and 894 us.
struct GFrag {
  double v[2][4];  // [sub-block][step]
};

// Lane index as a new value at each call: what is formed from it is computed
// where it is used.  The compiler otherwise forms it once for all the loops
// below, and then spills in them.
__device__ __forceinline__ int gemm_lane() {
  int l = threadIdx.x & 63;
  asm volatile("" : "+v"(l));
  return l;
}

// The loads address a wave-uniform pointer plus 32-bit lane offsets (bytes), so
// that a stream takes at most two registers per lane.
struct GStream {
  const char* p;  // wave-uniform, at k = 0 of the K range
  int64_t ld;     // bytes
  uint32_t off[2];
};

template <bool KC>
__device__ __forceinline__ GStream stream_at(const double* p, int64_t ld) {
  const int lane = gemm_lane(), li = lane & 15, lk = lane >> 4;
  GStream s;
  s.p = reinterpret_cast<const char*>(p);
  s.ld = ld * 8;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    s.off[i] = KC ? (uint32_t)(2 * (li & ~1)) * (uint32_t)(ld * 8) + 64 * (li & 1) + 16 * lk
                  : (uint32_t)(2 * lk + i) * (uint32_t)(ld * 8) + 16 * li;
  return s;
}

template <bool KC>
__device__ __forceinline__ void frag_load(const GStream& st, int k0, GFrag& f) {
  if (KC) {
    // load t: row 4 (li / 2) + t, k = 8 (li % 2) + 2 lk and the next
    const char* p = st.p + (int64_t)k0 * 8;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const dbl2u x = *reinterpret_cast<const dbl2u*>(p + t * st.ld + st.off[0]);
      f.v[t & 1][2 * (t >> 1)] = x.x;
      f.v[t & 1][2 * (t >> 1) + 1] = x.y;
    }
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const char* p = st.p + (int64_t)(k0 + 8 * h) * st.ld;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const dbl2u x = *reinterpret_cast<const dbl2u*>(p + st.off[i]);
        f.v[0][2 * h + i] = x.x;
        f.v[1][2 * h + i] = x.y;
      }
    }
  }
}

// Even lanes keep x and get y from the odd neighbour's x; odd lanes keep y and
// get x from the even neighbour's y.  One select per 32 bits, which takes one of
// its operands from the other lane (as a lane read and a select each, B
// transposed took 600 us); the wait states in front of a DPP read, and of an
// MFMA that reads the result, are written out, since the compiler does not track
// them into and out of an asm statement.
#define ROCBTA_SEL(d, n, o, q) \
  "v_cndmask_b32_dpp " d ", " n ", " o ", vcc quad_perm:[" q "] row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void pair_trade(double& x0, double& x1, double& y0, double& y1) {
  constexpr uint64_t even = 0x5555555555555555ull;
  const uint64_t u[4] = {__builtin_bit_cast(uint64_t, x0), __builtin_bit_cast(uint64_t, x1),
                         __builtin_bit_cast(uint64_t, y0), __builtin_bit_cast(uint64_t, y1)};
  uint32_t x[4], y[4], a[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    x[w] = (uint32_t)(u[w >> 1] >> (32 * (w & 1)));
    y[w] = (uint32_t)(u[2 + (w >> 1)] >> (32 * (w & 1)));
  }
  asm("s_mov_b64 vcc, %12\n\ts_nop 0\n\t" ROCBTA_SEL("%0", "%4", "%8", "0,0,2,2")
          ROCBTA_SEL("%1", "%5", "%9", "0,0,2,2") ROCBTA_SEL("%2", "%6", "%10", "0,0,2,2")
              ROCBTA_SEL("%3", "%7", "%11", "0,0,2,2") "s_nop 1"
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3])
      : "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]),
        "s"(even)
      : "vcc");
  asm("s_mov_b64 vcc, %8\n\ts_nop 0\n\t" ROCBTA_SEL("%0", "%4", "%0", "1,1,3,3")
          ROCBTA_SEL("%1", "%5", "%1", "1,1,3,3") ROCBTA_SEL("%2", "%6", "%2", "1,1,3,3")
              ROCBTA_SEL("%3", "%7", "%3", "1,1,3,3") "s_nop 1"
      : "+&v"(y[0]), "+&v"(y[1]), "+&v"(y[2]), "+&v"(y[3])
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "s"(~even)
      : "vcc");
  x0 = __builtin_bit_cast(double, ((uint64_t)a[1] << 32) | a[0]);
  x1 = __builtin_bit_cast(double, ((uint64_t)a[3] << 32) | a[2]);
  y0 = __builtin_bit_cast(double, ((uint64_t)y[1] << 32) | y[0]);
  y1 = __builtin_bit_cast(double, ((uint64_t)y[3] << 32) | y[2]);
}
#undef ROCBTA_SEL

// A group as KC loaded it to the layout of the MFMA steps.
template <bool KC>
__device__ __forceinline__ void frag_trade(GFrag& f) {
  if (!KC) return;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    pair_trade(f.v[i][0], f.v[i][1], f.v[i][2], f.v[i][3]);
}

// Blocks past the edge of C and a last partial group: loads without lane tests,
// two groups in flight.  Rows past the edge read row r_ok - 1 (what they give is
// not stored), so that every load has a valid address.  Such a block runs as long
// as the full ones beside it and so must not wait for each load: one 1100^3
// product with FP32 operands takes 58 us, 91 with tested loads used at once.
struct GEdge {
  const double* p[2];  // of row 2 li + i
  int64_t ld;
};
template <bool KC>
__device__ __forceinline__ GEdge edge_at(const double* p, int64_t ld, int r_ok) {
  const int li = gemm_lane() & 15;
  GEdge e;
  e.ld = ld;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = min(2 * li + i, r_ok - 1);
    e.p[i] = p + (KC ? (int64_t)r * ld : (int64_t)r);
  }
  return e;
}
// A group in the layout of the MFMA steps, zeros from index k_ok on (k0 < k_ok).
template <bool KC>
__device__ __forceinline__ void frag_load_edge(const GEdge& e, int k0, int k_ok, GFrag& f) {
  const int lk = gemm_lane() >> 4;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int k = k0 + 8 * (s >> 1) + 2 * lk + (s & 1), kc = min(k, k_ok - 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const double v = e.p[i][KC ? (int64_t)kc : (int64_t)kc * e.ld];
      f.v[i][s] = k < k_ok ? v : 0.0;
    }
  }
}

template <typename ACC>
__device__ __forceinline__ void frag_mfma(const GFrag& a, const GFrag& b, ACC (&acc)[2][2]) {
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma_acc(a.v[i][s], b.v[j][s], acc[i][j]);
}

// acc += op(A) op(B) of the wave's 32 x 32 block over the groups g = g0, g0 + gs,
// ... of 16 k in [0, ke); A and B point at the block's first row / column.
// Full blocks keep GPF groups in flight; blocks past the edge of C and a last
// partial group take the checked loads.
template <bool AK, bool BK, typename ACC>
__device__ __forceinline__ void gemm_wave(const double* A, int64_t lda, const double* B, int64_t ldb,
                                          int kb, int ke, int rows, int cols, int g0, int gs,
                                          ACC (&acc)[2][2]) {
  // groups without checks: full blocks whose lane offsets fit in 32 bits
  const bool fits = lda < (1 << 24) && ldb < (1 << 24);
  const int full = rows >= GW && cols >= GW && fits ? (ke - kb) / GK : 0;
  int g = g0;
  if (g < full) {
    const GStream sa = stream_at<AK>(A, lda), sb = stream_at<BK>(B, ldb);
    GFrag a[GPF], b[GPF];
#pragma unroll
    for (int u = 0; u < GPF; ++u)
      if (g + u * gs < full) {
        frag_load<AK>(sa, kb + (g + u * gs) * GK, a[u]);
        frag_load<BK>(sb, kb + (g + u * gs) * GK, b[u]);
      }
    while (g < full) {
#pragma unroll
      for (int u = 0; u < GPF; ++u) {
        if (g >= full) break;
        frag_trade<AK>(a[u]);
        frag_trade<BK>(b[u]);
        frag_mfma(a[u], b[u], acc);
        if (g + GPF * gs < full) {
          frag_load<AK>(sa, kb + (g + GPF * gs) * GK, a[u]);
          frag_load<BK>(sb, kb + (g + GPF * gs) * GK, b[u]);
        }
        g += gs;
      }
    }
  }
  if (kb + g * GK >= ke) return;
  const GEdge ea = edge_at<AK>(A, lda, rows), eb = edge_at<BK>(B, ldb, cols);
  GFrag a[2], b[2];
  frag_load_edge<AK>(ea, kb + g * GK, ke, a[0]);
  frag_load_edge<BK>(eb, kb + g * GK, ke, b[0]);
  for (bool more = true; more;) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (!more) break;
      g += gs;
      more = kb + g * GK < ke;
      if (more) {
        frag_load_edge<AK>(ea, kb + g * GK, ke, a[1 - u]);
        frag_load_edge<BK>(eb, kb + g * GK, ke, b[1 - u]);
      }
      frag_mfma(a[u], b[u], acc);
    }
  }
}

// K range of a term for the block at (m0, n0), restricted by the triangular
// shape of its operands.
__device__ __forceinline__ void gemm_k_range(const GemmTerm& t, int m0, int n0, int& kbeg,
                                             int& kend) {
  kbeg = 0;
  kend = t.K;
  if (t.triA == TRI_LOWER) kend = min(kend, m0 + GW);
  if (t.triA == TRI_UPPER) kbeg = max(kbeg, m0);
  if (t.triB == TRI_LOWER) kbeg = max(kbeg, n0);
  if (t.triB == TRI_UPPER) kend = min(kend, n0 + GW);
}

// One term of the wave's block; `at`: groups dealt to the waves before.  Returns
// whether the wave has one.
template <typename ACC>
__device__ __forceinline__ bool gemm_term(const GemmTerm& t, int b1, int b2, int M, int N, int m0,
                                          int n0, int wk, int gs, int& at, ACC (&acc)[2][2]) {
  int kb, ke;
  gemm_k_range(t, m0, n0, kb, ke);
  const int g0 = (wk - at) & (gs - 1);
  at += max(ke - kb + GK - 1, 0) / GK;
  if (kb + g0 * GK >= ke) return false;
  const double* A = t.A + b1 * t.sA1 + b2 * t.sA2 + (t.transA ? m0 : (int64_t)m0 * t.lda);
  const double* B = t.B + b1 * t.sB1 + b2 * t.sB2 + (t.transB ? (int64_t)n0 * t.ldb : n0);
  const int rows = M - m0, cols = N - n0;
  if (!t.transA && !t.transB)
    gemm_wave<true, false>(A, t.lda, B, t.ldb, kb, ke, rows, cols, g0, gs, acc);
  else if (!t.transA)
    gemm_wave<true, true>(A, t.lda, B, t.ldb, kb, ke, rows, cols, g0, gs, acc);
  else if (!t.transB)
    gemm_wave<false, false>(A, t.lda, B, t.ldb, kb, ke, rows, cols, g0, gs, acc);
  else
    gemm_wave<false, true>(A, t.lda, B, t.ldb, kb, ke, rows, cols, g0, gs, acc);
  return true;
}

// Sum of the two terms over the wave's share of K, to its LDS block: the groups
// of both are dealt in turn to the gs waves.  The terms' alphas are not applied
// to the operands: the block holds the sum in units of the last term's alpha
// (term 0's share is scaled by the quotient r0, exact for the +-1 in use), and the
// epilogue multiplies by it.  A second term with alpha 0 is skipped.  Each term
// starts from zero: with the accumulators carried from one to the next the
// second one's loops spill (four 1024^3 problems of two terms with B transposed:
// 432 us, 290 so).
template <typename ACC>
__device__ __forceinline__ void gemm_wave_block(const GemmProblem& P, const GemmTerm& t0,
                                                const GemmTerm& t1, bool two, double r0, int b1, int b2,
                                                int m0, int n0, int wk, int gs, double* part) {
  const bool in = m0 < P.M && n0 < P.N && P.nterms > 0;
  int at = 0;
  auto one = [&](const GemmTerm& term, int t) {
    ACC acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = ACC{0, 0, 0, 0};
    const bool has = in && gemm_term(term, b1, b2, P.M, P.N, m0, n0, wk, gs, at, acc);
    if (t && !has) return;
    const int lane = gemm_lane();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        dbl2* p = reinterpret_cast<dbl2*>(part + (2 * acc_row(acc[i][0], lane, r) + i) * GP +
                                          2 * acc_col(lane));
        dbl2 x;
        x.x = (double)acc[i][0][r];
        x.y = (double)acc[i][1][r];
        *p = t ? *p + x : x * r0;
      }
  };
  one(t0, 0);
  if (two) one(t1, 1);
}

// Tile `tile` (global index) of problem P: W x W blocks of 32 x 32, the K
// groups of each dealt to 8 / W^2 waves in turn, whose blocks are summed in
// wave order.
template <int W>
__device__ __forceinline__ void gemm_tile(const GemmProblem& P, int tile, double* lds) {
  constexpr int TS = GW * W, WK = GT_WAVES / (W * W);
  // tile rows per group of the grouped tile order (below)
  constexpr int GROUP_M = 8 / W;
  int local = tile - P.tile_begin;
  const int per_batch =
      P.lower_packed ? P.tiles_m * (P.tiles_m + 1) / 2 : P.tiles_m * P.tiles_n;
  const int bidx = local / per_batch;
  local -= bidx * per_batch;
  const int b1 = bidx % P.batch1, b2 = bidx / P.batch1;
  int tm, tn;
  if (P.lower_packed) {  // local = tm (tm + 1) / 2 + tn, 0 <= tn <= tm
    tm = (int)((__builtin_sqrtf(8.0f * (float)local + 1.0f) - 1.0f) * 0.5f);
    while ((tm + 1) * (tm + 2) / 2 <= local) ++tm;
    while (tm * (tm + 1) / 2 > local) --tm;
    tn = local - tm * (tm + 1) / 2;
  } else {
    // grouped order: GROUP_M tile rows at a time, column-major within the
    // group, so that a run of consecutive tiles (one XCD's share, see
    // xcd_tile) is a block of rows x columns sharing both operand panels
    const int first_m = (local / (GROUP_M * P.tiles_n)) * GROUP_M;
    const int rows = min(GROUP_M, P.tiles_m - first_m);
    const int within = local - first_m * P.tiles_n;
    tm = first_m + within % rows;
    tn = within / rows;
  }
  const int m0 = tm * TS, n0 = tn * TS;
  if (P.uplo == TRI_LOWER && n0 > m0 + TS - 1) return;
  if (P.uplo == TRI_UPPER && m0 > n0 + TS - 1) return;
  // read here, by scalar loads: after the first store (to LDS) they would be vector
  // loads, a round trip each
  const GemmTerm t0 = P.t[0], t1 = P.t[1];
  const int M = P.M, N = P.N, uplo = P.uplo, mirror = P.mirror;
  const int64_t ldc = P.ldc;
  const double beta = P.beta;
  double* const C = P.C + b1 * P.sC1 + b2 * P.sC2;
  const bool two = P.nterms == 2 && t1.alpha != 0.0;
  const double a_ref = two ? t1.alpha : t0.alpha;
  const double r0 = two ? t0.alpha / a_ref : 1.0;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave % WK, wb = wave / WK, wm = m0 + GW * (wb / W), wn = n0 + GW * (wb % W);
  if (P.f32)
    gemm_wave_block<f32x4>(P, t0, t1, two, r0, b1, b2, wm, wn, wk, WK, lds + wave * GW * GP);
  else
    gemm_wave_block<f64x4>(P, t0, t1, two, r0, b1, b2, wm, wn, wk, WK, lds + wave * GW * GP);
  __syncthreads();  // every operand has been read: C may now be written

  // thread: two adjacent columns of W * W rows (one per 32 x 32 block)
  const int rr = threadIdx.x >> 4, cc = 2 * (threadIdx.x & 15);
#pragma unroll
  for (int blk = 0; blk < W * W; ++blk) {
    double* part = lds + blk * WK * GW * GP + rr * GP + cc;
    dbl2 s = *reinterpret_cast<const dbl2*>(part);
#pragma unroll
    for (int q = 1; q < WK; ++q) s += *reinterpret_cast<const dbl2*>(part + q * GW * GP);
    const int row = m0 + GW * (blk / W) + rr, col = n0 + GW * (blk % W) + cc;
    double* c = C + (int64_t)row * ldc + col;
    const bool full = row < M && col + 1 < N && uplo == TRI_NONE;
    s *= a_ref;
    if (full) {
      if (beta != 0.0) s += beta * (dbl2)*reinterpret_cast<const dbl2u*>(c);
      *reinterpret_cast<dbl2u*>(c) = s;
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (row >= M || col + e >= N) continue;
        if (uplo == TRI_LOWER && col + e > row) continue;
        if (uplo == TRI_UPPER && col + e < row) continue;
        double v = e ? s.y : s.x;
        if (beta != 0.0) v += beta * c[e];
        c[e] = v;
        if (e) s.y = v; else s.x = v;
      }
    }
    if (mirror) *reinterpret_cast<dbl2*>(part) = s;
  }
  if (!mirror) return;
  // the transposed entries, read back from LDS so that they are stored by rows
  __syncthreads();
#pragma unroll
  for (int blk = 0; blk < W * W; ++blk) {
    const double* part = lds + blk * WK * GW * GP;
    // element (cc + e, rr) of the block goes to C[col of it][row of it]
    const int col = n0 + GW * (blk % W) + rr;
    double* c = C + (int64_t)col * ldc;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int row = m0 + GW * (blk / W) + cc + e;
      if (row < M && col < row) c[row] = part[(cc + e) * GP + rr];
    }
  }
}

// Workgroup -> tile order.  Workgroups are dealt to the 8 XCDs round-robin
// (workgroup w runs on XCD w mod 8), each with its own L2.  Giving XCD x a
// contiguous range of tile indices makes the workgroups of one XCD share
// their operand panels in that L2 instead of every XCD streaming every panel.
// A bijection of [0, ntiles), so any dispatch order stays correct.
constexpr int N_XCD = 8;
__device__ __forceinline__ int xcd_tile(int w, int ntiles) {
  const int q = ntiles / N_XCD, r = ntiles % N_XCD;
  const int x = w % N_XCD, i = w / N_XCD;
  return x * q + min(x, r) + i;
}

template <int W>
__global__ void __launch_bounds__(GT_THREADS, 4) gemm_group_kernel(GemmGroup g) {
  __shared__ __attribute__((aligned(16))) double lds[GT_WAVES * GW * GP];
  const int tile = xcd_tile(blockIdx.x, g.total_tiles);
  int pi = 0;
  while (pi + 1 < g.nprob && tile >= g.p[pi + 1].tile_begin) ++pi;
  gemm_tile<W>(g.p[pi], tile, lds);
}

// The same over a device array of problems (sorted by tile_begin): used by the
// batched plans, whose launch lists are built once and replayed.
template <int W>
__global__ void __launch_bounds__(GT_THREADS, 4) gemm_list_kernel(const GemmProblem* probs,
                                                                  int nprob) {
  __shared__ __attribute__((aligned(16))) double lds[GT_WAVES * GW * GP];
  const int tile = blockIdx.x;
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (probs[mid].tile_begin <= tile) lo = mid; else hi = mid - 1;
  }
  gemm_tile<W>(probs[lo], tile, lds);
}

}  // namespace rocbta
