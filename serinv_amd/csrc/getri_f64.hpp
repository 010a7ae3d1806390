// General (non-symmetric) inverse of an m x m block by in-place Gauss-Jordan
// elimination over 64-wide pivot tiles without pivoting, for the diagonally
// dominant blocks of the non-SPD (ddbt*) routines, where elimination without
// row exchanges is stable.  Step k, with P = A_kk^{-1}:
//   A_kk <- P;  A_kj <- P A_kj;  A_ij <- A_ij - A_ik (P A_kj);  A_ik <- -A_ik P.
// One launch per step, one workgroup per tile, from one copy of the matrix to
// the other (a step reads tiles that other workgroups write).  Every workgroup
// inverts A_kk and forms P A_kj for itself: the step is bound by the latency
// of that chain, and a launch costs less than a hand-off of P and of the row
// panel between workgroups would.  It takes the place of a launch for P, one
// for the row panel, one for the update and one for the column panel.
//
// The tile inverse (lds_getri64) is the same elimination over 16-wide pivot
// blocks in LDS: the 16 x 16 pivot block by one wave in registers, the panels
// and the update on MFMA.
#pragma once
#include "common.hpp"
#include "tile_f64.hpp"
#include "pobtaf_chain.hpp"

namespace rocbta {

// v[j] -= v[j](lane K of the row) * g for j = J0 .. J0 + N - 1 (not K).
#define ROCBTA_GJ(x) \
  "v_fmac_f64_dpp " x ", -" x ", %[g] row_newbcast:%[k] row_mask:0xf bank_mask:0xf\n\t"
#define ROCBTA_IN : [g] "v"(g), [k] "n"(K)
template <int K, int J0, int N>
__device__ __forceinline__ void gj_row_fmac(double (&v)[PW], double g) {
  if constexpr (N >= 4) {
    asm volatile("s_nop 1\n\t" ROCBTA_GJ("%0") ROCBTA_GJ("%1") ROCBTA_GJ("%2") ROCBTA_GJ("%3")
                 : "+v"(v[J0]), "+v"(v[J0 + 1]), "+v"(v[J0 + 2]), "+v"(v[J0 + 3]) ROCBTA_IN);
    gj_row_fmac<K, J0 + 4, N - 4>(v, g);
  } else if constexpr (N >= 2) {
    asm volatile("s_nop 1\n\t" ROCBTA_GJ("%0") ROCBTA_GJ("%1")
                 : "+v"(v[J0]), "+v"(v[J0 + 1]) ROCBTA_IN);
    gj_row_fmac<K, J0 + 2, N - 2>(v, g);
  } else if constexpr (N == 1) {
    asm volatile("s_nop 1\n\t" ROCBTA_GJ("%0") : "+v"(v[J0]) ROCBTA_IN);
  }
}
#undef ROCBTA_IN
#undef ROCBTA_GJ

// Gauss-Jordan steps K .. 15 of the 16 x 16 block in v (lane li of every
// 16-lane row: matrix row li); rp: reciprocal of pivot K.  The pivot row is
// left unscaled; its factor is kept in sc (lane K) and applied to the whole
// row at the end, which is the same elimination because every step is linear
// in each row.
template <int K>
__device__ __forceinline__ void gj_columns(double (&v)[PW], double rp, double& sc, int li) {
  if constexpr (K < PW) {
    const double g = li == K ? 0.0 : v[K] * rp;
    double rn = 0.0;
    if constexpr (K + 1 < PW) {  // the next pivot first
      gj_row_fmac<K, K + 1, 1>(v, g);
      rn = 1.0 / row_bcast<K + 1>(v[K + 1]);
      gj_row_fmac<K, K + 2, PW - K - 2>(v, g);
    }
    gj_row_fmac<K, 0, K>(v, g);
    v[K] = li == K ? 1.0 : -g;
    sc = li == K ? rp : sc;
    gj_columns<K + 1>(v, rn, sc, li);
  }
}

// S (64 x 64, row pitch LD, in LDS) <- S^{-1}; Pk: 16 x 17 scratch.  256
// threads; the caller's barrier precedes it, and it ends with one.
template <int LD>
__device__ __forceinline__ void lds_getri64(double* S, double* Pk) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  constexpr int PL = 17;
#pragma unroll 1
  for (int kb = 0; kb < 4; ++kb) {
    const int k0 = 16 * kb;
    if (wave == 0) {
      double v[PW], sc = 1.0;
#pragma unroll
      for (int j = 0; j < PW; ++j) v[j] = S[(k0 + li) * LD + k0 + j];
      gj_columns<0>(v, 1.0 / row_bcast<0>(v[0]), sc, li);
      if (lane < 16) {
#pragma unroll
        for (int j = 0; j < PW; ++j) Pk[li * PL + j] = v[j] * sc;
      }
    }
    __syncthreads();
    if (wave < 3) {  // row panel: the wave's block column jb
      const int jb = wave + (wave >= kb ? 1 : 0);
      f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int kk = 0; kk < 16; kk += 4)
        acc = mfma_f64(Pk[li * PL + kk + lk], S[(k0 + kk + lk) * LD + 16 * jb + li], acc);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[(k0 + acc_row_f64(lane, r)) * LD + 16 * jb + li] = acc[r];
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) S[(k0 + 4 * r + lk) * LD + k0 + li] = Pk[(4 * r + lk) * PL + li];
    }
    __syncthreads();
    if (wave < 3) {  // the wave's block row ib: update, then its column block
      const int ib = wave + (wave >= kb ? 1 : 0);
      double c[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) c[r] = -S[(16 * ib + li) * LD + k0 + 4 * r + lk];
      f64x4 acc[4];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[jb][r] = jb == kb ? 0.0 : S[(16 * ib + acc_row_f64(lane, r)) * LD + 16 * jb + li];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
          acc[jb] = mfma_f64(c[kk], S[(k0 + 4 * kk + lk) * LD + 16 * jb + li], acc[jb]);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[(16 * ib + acc_row_f64(lane, r)) * LD + 16 * jb + li] = acc[jb][r];
    }
    __syncthreads();
  }
}

// acc += sgn * A B over k in [0, 64): A = XA[m][k], B = XB[k][n] (pitch KP).
__device__ __forceinline__ void gj_mfma(const double* XA, const double* XB, f64x4 (&acc)[2][2],
                                        double sgn) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll 4
  for (int kk = 0; kk < CT; kk += 4) {
    const double a0 = sgn * XA[(wm + li) * KP + kk + lk], a1 = sgn * XA[(wm + 16 + li) * KP + kk + lk];
    const double b0 = XB[(kk + lk) * KP + wn + li], b1 = XB[(kk + lk) * KP + wn + 16 + li];
    acc[0][0] = mfma_f64(a0, b0, acc[0][0]);
    acc[0][1] = mfma_f64(a0, b1, acc[0][1]);
    acc[1][0] = mfma_f64(a1, b0, acc[1][0]);
    acc[1][1] = mfma_f64(a1, b1, acc[1][1]);
  }
}

// Step k of the inverse: tile (blockIdx.x % T, blockIdx.x / T) of dst from src.
// With T == 1 src and dst may be the same.  Partial edge tiles are padded with
// the identity, which the elimination leaves alone.
__global__ void __launch_bounds__(CH_THREADS) block_getri_kernel(const double* src, int64_t lds_,
                                                                 double* dst, int64_t ldd, int m,
                                                                 int T, int k) {
  __shared__ __attribute__((aligned(16))) double S[CT * KP], XA[CT * KP], XB[CT * KP], Pk[16 * 17];
  const int i = blockIdx.x / T, j = blockIdx.x % T;
  const int tid = threadIdx.x;
  auto tile = [&](const double* p, int64_t ld, int r, int c) {
    return CTile{const_cast<double*>(p) + (int64_t)r * CT * ld + (int64_t)c * CT, ld,
                 cmin(CT, m - r * CT), cmin(CT, m - c * CT)};
  };
  TileRegs16 rk, ra, rb;
  f64x4 own[2][2];
  tile_load16(tile(src, lds_, k, k), rk);
  if (i != k) tile_load16(tile(src, lds_, i, k), ra);
  if (j != k) tile_load16(tile(src, lds_, k, j), rb);
  if (i != k && j != k)
    cacc_load(tile(src, lds_, i, j), own);
  else
    cacc_zero(own);
  tile_store16(rk, S);
  if (i != k) tile_store16(ra, XA);
  if (j != k) tile_store16(rb, XB);
  __syncthreads();
  const int mk = cmin(CT, m - k * CT);
  if (tid >= mk && tid < CT) S[tid * KP + tid] = 1.0;
  __syncthreads();
  lds_getri64<KP>(S, Pk);
  const CTile out = tile(dst, ldd, i, j);
  if (i == k && j == k) {
    lds_tile_store(S, KP, out);
    return;
  }
  if (j == k) {
    gj_mfma(XA, S, own, -1.0);  // -A_ik P
  } else {
    f64x4 row[2][2];
    cacc_zero(row);
    gj_mfma(S, XB, row, 1.0);  // P A_kj
    if (i == k) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) own[x][y] = row[x][y];
    } else {
      __syncthreads();  // XB and S have been read
      cacc_to_lds(row, XB, KP);
      __syncthreads();
      gj_mfma(XA, XB, own, -1.0);
    }
  }
  __syncthreads();
  cacc_to_lds(own, S, KP);
  __syncthreads();
  lds_tile_store(S, KP, out);
}

// Inverse of one tile (m <= 64), in place or to P.
__global__ void __launch_bounds__(CH_THREADS) tile_getri_kernel(const double* A, int64_t lda, int m,
                                                               double* P, int64_t ldp) {
  __shared__ __attribute__((aligned(16))) double S[CT * KP], Pk[16 * 17];
  const int tid = threadIdx.x;
  TileRegs16 r;
  tile_load16(CTile{const_cast<double*>(A), lda, m, m}, r);
  tile_store16(r, S);
  __syncthreads();
  if (tid >= m && tid < CT) S[tid * KP + tid] = 1.0;
  __syncthreads();
  lds_getri64<KP>(S, Pk);
  lds_tile_store(S, KP, CTile{P, ldp, m, m});
}

}  // namespace rocbta
