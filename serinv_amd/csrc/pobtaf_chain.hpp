// Persistent block Cholesky of an SPD BTA matrix (pobtaf) on gfx950:
// one CHAIN workgroup walks the diagonal tiles, HELPER workgroups do the rest.
//
// The reference recurrence (src/serinv/algs/pobtaf.py:115-183) is evaluated on
// 64x64 tiles.  Tiles are addressed in global tile coordinates: tile row /
// column g = i * nt + c is tile c of block i (nt = ceil(b / 64)); the band of
// tile column j (block jb) holds rows j .. (jb + 2) * nt - 1 (the rest of D_jb
// and all of L_{jb+1,jb}), plus the arrow tile of R_jb.  L(r, k) denotes a
// finished factor tile.
//
// Chain workgroup, step g (strictly sequential):
//   D(g,g) <- PD(g) - L(g,g-1) L(g,g-1)^T       (L(g,g-1) kept in LDS)
//   L(g,g) = chol(D(g,g)), Linv(g) = L(g,g)^{-1}  -> published
//   L(g+1,g) = PX(g) Linv(g)^T                    -> published, kept in LDS
// where PD(g) = D(g,g) minus the products of all columns k < g-1 and
// PX(g) = X(g+1,g) minus the products of all columns k < g are prepared by
// helpers.  Helper tasks:
//   TRSM(r, j), r >= j + 2 : X(r,j) - sum_k L(r,k) L(j,k)^T, then * Linv(j)^T
//   ARR(j, q)              : the same for arrow tile q (64 arrow rows) of column j
//   PX(g), PD(g)           : the partial sums above (stored in place)
//   TIPP(i)                : P_i = R_i R_i^T;  TIP: chol(T - P_0 - ... - P_{n-1})
//                            (arrows of one tile; wider ones leave the tip to the caller)
// Helper tasks are taken from an atomic queue organised in stages; stage h
// holds the tasks that need chain outputs of steps <= h - 1 only, and inside
// a stage every task only waits on earlier slots.  The chain step g needs
// PD(g) (stage g-1) and PX(g) (stage g), so no wait can cycle.  Every wait is
// bounded: an overrun sets info = -1 and makes all later waits return.
//
// Memory ordering: tiles are published with an agent-scope release before
// the flag store; waiters poll relaxed and issue one agent-scope acquire.
#pragma once
#include "common.hpp"
#include "tile_f64.hpp"

namespace rocbta {

constexpr int CT = 64;          // tile size
constexpr int CH_THREADS = 256;
constexpr int KP = CT + 2;      // pitch of K-contiguous LDS tiles (doubles)

struct PobtafChain {
  double* D;
  double* L;
  double* R;
  double* T;
  int n, b, a, nt;
  int na;       // arrow tiles of a column: ceil(a / 64)
  int NT;       // number of diagonal tiles (n * nt)
  int slots;    // helper slots per stage
  int nstages;  // NT + 2
  int ntasks;   // nstages * slots
  int* counter;  // helper queue head
  int* claim;    // chain claim ticket
  int* hflags;   // helper task flags
  int* cflags;   // chain flags: [2g] Linv(g) ready, [2g+1] L(g+1,g) ready
  int* info;
  int* chain_cu;  // 1 + hardware CU key of the chain workgroup (0 until known)
  double* linv;   // NT * 64 * 64
  double* tipp;   // n * a * a
  double* tip_inv;  // optional (batched plans): L_T^{-1} as a 64 x 64 tile
  long long spin_limit;
  // Mixed precision: the tile products (trsm, syrk/gemm updates) round their
  // FP64 operands to FP32 and accumulate in FP32 MFMA; the tiles stay FP64
  // in memory and the diagonal potrf / trtri and the tip run in FP64.
  int f32;
  // Diagnostic timeline (nullptr normally): 100 MHz timestamps, CHAIN_TRACE_EV
  // per chain step g at trace[CHAIN_TRACE_EV * g + e], see chain_trace.
  long long* trace;
};

// Timeline events of chain step g (diagnostic builds of a run):
//   0 step start, 1 factorization done, 2 Linv(g) released, PX(g)/PD(g+1)
//   staged, 3 L(g+1,g) complete, 5 step end, 6 PX(g) published (by its helper), 7 L(g+2,g) published (by its helper).
constexpr int CHAIN_TRACE_EV = 8;
__device__ __forceinline__ void chain_trace(const PobtafChain& P, int g, int e) {
  if (P.trace && threadIdx.x == 0)
    P.trace[CHAIN_TRACE_EV * g + e] = (long long)__builtin_amdgcn_s_memrealtime();
}

// Hardware key of the CU running the calling wave: XCC id and the
// SE/SH/CU fields of HW_ID.
__device__ __forceinline__ int hw_cu_key() {
  const unsigned hw = __builtin_amdgcn_s_getreg((31 << 11) | (0 << 6) | 4);     // HW_ID
  const unsigned xcc = __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20);    // XCC_ID
  return (int)(((xcc & 15u) << 8) | ((hw >> 8) & 0xffu));
}

struct CTile {
  double* p;
  int64_t ld;
  int rows, cols;
};

enum ChainKind { HK_NOOP = 0, HK_TRSM = 1, HK_PX = 2, HK_PD = 3, HK_ARR = 4, HK_TIPP = 5, HK_TIP = 6 };

__host__ __device__ __forceinline__ int cmin(int x, int y) { return x < y ? x : y; }
__host__ __device__ __forceinline__ int cmax(int x, int y) { return x > y ? x : y; }

// exclusive end of the band rows of tile column j
__host__ __device__ __forceinline__ int band_end(const PobtafChain& P, int j) {
  const int jb = j / P.nt;
  return (jb < P.n - 1) ? (jb + 2) * P.nt : (jb + 1) * P.nt;
}
// first contributing column for a row of block rb
__host__ __device__ __forceinline__ int kmin_of(const PobtafChain& P, int rb) {
  return cmax(0, (rb - 1) * P.nt);
}

__host__ __device__ __forceinline__ CTile tile_g(const PobtafChain& P, int r, int j) {
  const int jb = j / P.nt, jc = j % P.nt, rb = r / P.nt, rc = r % P.nt;
  const int64_t b = P.b;
  double* base = (rb == jb) ? P.D : P.L;
  return {base + (int64_t)jb * b * b + (int64_t)rc * CT * b + (int64_t)jc * CT, b,
          cmin(CT, P.b - rc * CT), cmin(CT, P.b - jc * CT)};
}
// Strict-upper D tile (jc, rc) that mirrors the lower tile (r, j) of the same
// block; the factor has zeros there.
__host__ __device__ __forceinline__ CTile tile_mirror(const PobtafChain& P, int r, int j) {
  const int jb = j / P.nt, jc = j % P.nt, rc = r % P.nt;
  const int64_t b = P.b;
  return {P.D + (int64_t)jb * b * b + (int64_t)jc * CT * b + (int64_t)rc * CT, b,
          cmin(CT, P.b - jc * CT), cmin(CT, P.b - rc * CT)};
}
__host__ __device__ __forceinline__ CTile tile_arrow(const PobtafChain& P, int j, int q) {
  const int jb = j / P.nt, jc = j % P.nt;
  const int64_t b = P.b;
  return {P.R + ((int64_t)jb * P.a + q * CT) * b + (int64_t)jc * CT, b, cmin(CT, P.a - q * CT),
          cmin(CT, P.b - jc * CT)};
}

// ---------------------------------------------------------- task indexing
// slot layout of stage h (j = h - 1):
//   0             TRSM(j+2, j)
//   1             PX(h)
//   2             PD(h+1)
//   3 .. 3+2nt-1  TRSM(j+3+q, j)
//   3+2nt+q       ARR(j, q), q < na
//   slots - 1     TIPP(h/nt - 1) when h is a multiple of nt (na = 1)
// stage NT+1, slot 0: TIP (na = 1)
__host__ __device__ __forceinline__ int chain_slots(int nt, int na) { return 4 + 2 * nt + cmax(na, 1); }
__host__ __device__ __forceinline__ int t_trsm(const PobtafChain& P, int r, int j) {
  const int h = j + 1;
  return h * P.slots + ((r == j + 2) ? 0 : 3 + (r - (j + 3)));
}
__host__ __device__ __forceinline__ int t_px(const PobtafChain& P, int g) { return g * P.slots + 1; }
__host__ __device__ __forceinline__ int t_pd(const PobtafChain& P, int g) {
  return (g - 1) * P.slots + 2;
}
__host__ __device__ __forceinline__ int t_arr(const PobtafChain& P, int j, int q) {
  return (j + 1) * P.slots + 3 + 2 * P.nt + q;
}
__host__ __device__ __forceinline__ int t_tippc(const PobtafChain& P, int i) {
  return ((i + 1) * P.nt) * P.slots + P.slots - 1;
}
__host__ __device__ __forceinline__ int t_tipc(const PobtafChain& P) {
  return (P.NT + 1) * P.slots;
}

// Decode a helper task: kind, and (r, j) = output tile (TRSM), g in j (PX/PD),
// arrow tile r of column j (ARR), block i in j (TIPP).
__host__ __device__ __forceinline__ int chain_decode(const PobtafChain& P, int task, int& r,
                                                     int& j) {
  const int h = task / P.slots, slot = task % P.slots;
  r = 0;
  j = 0;
  if (h == P.NT + 1) return (slot == 0 && P.na == 1) ? HK_TIP : HK_NOOP;
  const int jj = h - 1;
  if (slot == 0) {
    if (jj >= 0 && jj + 2 < band_end(P, jj)) {
      r = jj + 2;
      j = jj;
      return HK_TRSM;
    }
    return HK_NOOP;
  }
  if (slot == 1) {
    if (h < P.NT && h + 1 < band_end(P, h)) {
      j = h;
      return HK_PX;
    }
    return HK_NOOP;
  }
  if (slot == 2) {
    if (h + 1 < P.NT) {
      j = h + 1;
      return HK_PD;
    }
    return HK_NOOP;
  }
  if (slot < 3 + 2 * P.nt) {
    const int rr = jj + 3 + (slot - 3);
    if (jj >= 0 && rr < band_end(P, jj)) {
      r = rr;
      j = jj;
      return HK_TRSM;
    }
    return HK_NOOP;
  }
  if (slot < 3 + 2 * P.nt + P.na) {
    if (jj >= 0) {
      r = slot - (3 + 2 * P.nt);
      j = jj;
      return HK_ARR;
    }
    return HK_NOOP;
  }
  if (slot == P.slots - 1 && P.na == 1 && h >= P.nt && h % P.nt == 0) {
    j = h / P.nt - 1;
    return HK_TIPP;
  }
  return HK_NOOP;
}

// Readiness flag of the factor tile (r, k), r > k (r < 0: arrow tile -1 - r).
__host__ __device__ __forceinline__ int* factor_flag(const PobtafChain& P, int r, int k) {
  if (r < 0) return P.hflags + t_arr(P, k, -1 - r);
  if (r == k + 1) return P.cflags + 2 * k + 1;
  return P.hflags + t_trsm(P, r, k);
}

// Contribution list of a helper task: columns k in [k0, k1) with operands
// A = factor tile (ra, k) (ra < 0: arrow tile -1 - ra) and B = factor tile (jb, k).
struct ContribRange {
  int ra, jb, k0, k1;
};
__host__ __device__ __forceinline__ ContribRange chain_contribs(const PobtafChain& P, int kind,
                                                               int r, int j) {
  switch (kind) {
    case HK_TRSM:
      return {r, j, kmin_of(P, r / P.nt), j};
    case HK_ARR:
      return {-1 - r, j, kmin_of(P, j / P.nt), j};
    case HK_PX:
      return {j + 1, j, kmin_of(P, (j + 1) / P.nt), j};
    case HK_PD:
      return {j, j, kmin_of(P, j / P.nt), j - 1};
    default:
      return {0, 0, 0, 0};
  }
}

// ---------------------------------------------------------------- flags
__device__ __forceinline__ bool chain_poll(const PobtafChain& P, const int* f, long long& spins) {
  while (__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
    if (++spins > P.spin_limit) return false;
    if ((spins & 255) == 0 &&
        __hip_atomic_load(P.info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < 0)
      return false;
    __builtin_amdgcn_s_sleep(1);
  }
  return true;
}

// Wait for flags fa (and fb if non-null); all threads return after an acquire.
__device__ __forceinline__ void chain_wait(const PobtafChain& P, const int* fa, const int* fb) {
  if (threadIdx.x == 0) {
    long long spins = 0;
    bool ok = chain_poll(P, fa, spins);
    if (ok && fb) ok = chain_poll(P, fb, spins);
    if (!ok) __hip_atomic_store(P.info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}

// The calling wave alone waits for fa (and fb if non-null), then acquires.
// All lanes poll the same address, so the loop is uniform; no barrier.
__device__ __forceinline__ void wave_wait(const PobtafChain& P, const int* fa, const int* fb) {
  long long spins = 0;
  bool ok = chain_poll(P, fa, spins);
  if (ok && fb) ok = chain_poll(P, fb, spins);
  if (!ok && (threadIdx.x & 63) == 0)
    __hip_atomic_store(P.info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

// Every wave waits for its own global stores to complete (s_waitcnt
// vmcnt(0)) before the barrier: a workgroup barrier does not wait for them,
// and the release by thread 0 (L2 write-back, then its own wave's counter)
// would otherwise miss stores of other waves still on their way to L2.
// With all of them in L2, thread 0's single release covers the tile.
__device__ __forceinline__ void wave_stores_done() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// The explicit wait after thread 0's release fence keeps the flag store
// behind the completion of the L2 write-back: with the counters already
// drained, the compiler otherwise emits no wait between the two.
__device__ __forceinline__ void chain_publish(int* f, int publisher = 0) {
  wave_stores_done();
  __syncthreads();
  if ((int)threadIdx.x == publisher) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    wave_stores_done();
    __hip_atomic_store(f, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ----------------------------------------------------------- tile movement
typedef double cdbl2 __attribute__((ext_vector_type(2)));
typedef double cdbl2u __attribute__((ext_vector_type(2), aligned(8)));  // any double address

// Thread t holds rows (t >> 5) + 8q (q = 0..7), columns 2*(t & 31) .. +1 of a
// 64x64 tile: each wave load instruction covers two whole 512-byte rows.
struct TileRegs16 {
  cdbl2 v[8];
};

__device__ __forceinline__ void tile_load16(const CTile& t, TileRegs16& x) {
  const int rs = threadIdx.x >> 5, c = (threadIdx.x & 31) * 2;
  if (t.rows == CT && t.cols == CT) {
#pragma unroll
    for (int q = 0; q < 8; ++q)
      x.v[q] = *reinterpret_cast<const cdbl2u*>(t.p + (int64_t)(rs + 8 * q) * t.ld + c);
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int row = rs + 8 * q;
      const double* src = t.p + (int64_t)row * t.ld + c;
      x.v[q].x = (row < t.rows && c < t.cols) ? src[0] : 0.0;
      x.v[q].y = (row < t.rows && c + 1 < t.cols) ? src[1] : 0.0;
    }
  }
}

// K-contiguous staging: X[row][k] with pitch KP (row = m or n index).
__device__ __forceinline__ void tile_store16(const TileRegs16& x, double* X) {
  const int rs = threadIdx.x >> 5, c = (threadIdx.x & 31) * 2;
#pragma unroll
  for (int q = 0; q < 8; ++q) *reinterpret_cast<cdbl2*>(X + (rs + 8 * q) * KP + c) = x.v[q];
}

// acc (+)= sgn * A B^T over k in [0, 64), A = XA[m][k], B = XB[n][k].
template <typename ACC>
__device__ __forceinline__ void mfma_abt(const double* XA, const double* XB, ACC (&acc)[2][2],
                                         double sgn, bool lower_only) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  if (lower_only && wn > wm) return;
  const int li = lane & 15, lk = lane >> 4;
  // operands double-buffered across k steps: the LDS reads of step kk + 4
  // are issued before the MFMAs of step kk
  double a[2][2], b[2][2];
  auto fetch = [&](int buf, int kk) {
    a[buf][0] = XA[(wm + li) * KP + kk + lk];
    a[buf][1] = XA[(wm + 16 + li) * KP + kk + lk];
    b[buf][0] = XB[(wn + li) * KP + kk + lk];
    b[buf][1] = XB[(wn + 16 + li) * KP + kk + lk];
  };
  fetch(0, 0);
#pragma unroll
  for (int kk = 0; kk < CT; kk += 4) {
    const int cur = (kk >> 2) & 1;
    if (kk + 4 < CT) fetch(cur ^ 1, kk + 4);
    __builtin_amdgcn_sched_barrier(0);
    const double a0 = sgn * a[cur][0], a1 = sgn * a[cur][1];
    acc[0][0] = mfma_acc(a0, b[cur][0], acc[0][0]);
    acc[0][1] = mfma_acc(a0, b[cur][1], acc[0][1]);
    acc[1][0] = mfma_acc(a1, b[cur][0], acc[1][0]);
    acc[1][1] = mfma_acc(a1, b[cur][1], acc[1][1]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// acc += a32 (an FP32 accumulator in the FP32 MFMA register layout),
// remapped through the 64 x 64 LDS scratch X (row pitch `pitch`).  X must be
// free once every wave arrives; the call starts and ends with a barrier.
__device__ __forceinline__ void acc32_add(const f32x4 (&a32)[2][2], f64x4 (&acc)[2][2], double* X,
                                          int pitch) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        X[(wm + i * 16 + acc_row_f32(lane, r)) * pitch + wn + j * 16 + acc_col(lane)] =
            (double)a32[i][j][r];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[i][j][r] += X[(wm + i * 16 + acc_row_f64(lane, r)) * pitch + wn + j * 16 + acc_col(lane)];
  __syncthreads();
}

__device__ __forceinline__ void cacc32_zero(f32x4 (&acc)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

__device__ __forceinline__ void cacc_zero(f64x4 (&acc)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
}

__device__ __forceinline__ void cacc_load(const CTile& t, f64x4 (&acc)[2][2]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wm + i * 16 + acc_row_f64(lane, r), col = wn + j * 16 + acc_col(lane);
        acc[i][j][r] = (row < t.rows && col < t.cols) ? t.p[(int64_t)row * t.ld + col] : 0.0;
      }
}

__device__ __forceinline__ void cacc_store(const CTile& t, const f64x4 (&acc)[2][2]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wm + i * 16 + acc_row_f64(lane, r), col = wn + j * 16 + acc_col(lane);
        if (row < t.rows && col < t.cols) t.p[(int64_t)row * t.ld + col] = acc[i][j][r];
      }
}

// Stage the accumulator in LDS: X[row * pitch + col] = acc(row, col).
__device__ __forceinline__ void cacc_to_lds(const f64x4 (&acc)[2][2], double* X, int pitch) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        X[(wm + i * 16 + acc_row_f64(lane, r)) * pitch + wn + j * 16 + acc_col(lane)] =
            acc[i][j][r];
}

// Store a tile staged in LDS (X[row * pitch + col]) to memory: each thread
// reads its 8 row pairs (rows rs + 8q, columns c, c + 1) first and then issues
// the stores, 16 bytes each for full tiles.
__device__ __forceinline__ void lds_tile_store(const double* X, int pitch, const CTile& t) {
  const int rs = threadIdx.x >> 5, c = (threadIdx.x & 31) * 2;
  cdbl2 v[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    v[q].x = X[(rs + 8 * q) * pitch + c];
    v[q].y = X[(rs + 8 * q) * pitch + c + 1];
  }
  double* dst = t.p + (int64_t)rs * t.ld + c;
  if (t.rows == CT && t.cols == CT) {
#pragma unroll
    for (int q = 0; q < 8; ++q) *reinterpret_cast<cdbl2u*>(dst + (int64_t)(8 * q) * t.ld) = v[q];
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (rs + 8 * q < t.rows && c < t.cols) dst[(int64_t)(8 * q) * t.ld] = v[q].x;
      if (rs + 8 * q < t.rows && c + 1 < t.cols) dst[(int64_t)(8 * q) * t.ld + 1] = v[q].y;
    }
  }
}

// Zero a whole tile (used for the strict-upper tiles of the D blocks).
__device__ __forceinline__ void tile_zero(const CTile& t) {
  for (int idx = threadIdx.x; idx < CT * CT; idx += CH_THREADS) {
    const int row = idx >> 6, col = idx & 63;
    if (row < t.rows && col < t.cols) t.p[(int64_t)row * t.ld + col] = 0.0;
  }
}

// ------------------------------------------------------------ helper work
// acc -= sum over the contribution range (A = factor tile (ra,k) or an arrow
// tile of column k, B = factor tile (jb,k)); operands prefetched one product ahead.
// TAG gives each kernel its own copy of the non-inlined workers, so that
// each copy sees a single kind of descriptor pointer (kernel argument or
// global array) and is optimised for it.
template <typename ACC>
__device__ __forceinline__ void helper_products(const PobtafChain& P, const ContribRange& cr,
                                                double sgn, bool lower_only, double* XA,
                                                double* XB, ACC (&acc)[2][2]) {
  TileRegs16 ra, rb;
  auto tileA = [&](int k) { return cr.ra < 0 ? tile_arrow(P, k, -1 - cr.ra) : tile_g(P, cr.ra, k); };
  __shared__ int s_ready;
  chain_wait(P, factor_flag(P, cr.ra, cr.k0), factor_flag(P, cr.jb, cr.k0));
  tile_load16(tileA(cr.k0), ra);
  tile_load16(tile_g(P, cr.jb, cr.k0), rb);
  for (int k = cr.k0;; ++k) {
    const bool more = k + 1 < cr.k1;
    __syncthreads();  // previous product done with XA / XB
    tile_store16(ra, XA);
    tile_store16(rb, XB);
    // The next contribution is prefetched only if its tiles are already
    // published (checked without waiting); otherwise this product runs
    // first and the wait follows it, so that the last product of a task is
    // not held behind the wait for it.
    if (threadIdx.x == 0) {
      int ready = 0;
      if (more &&
          __hip_atomic_load(factor_flag(P, cr.ra, k + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &&
          __hip_atomic_load(factor_flag(P, cr.jb, k + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        ready = 1;
      }
      s_ready = ready;
    }
    __syncthreads();
    const bool pre = more && s_ready;
    if (pre) {
      tile_load16(tileA(k + 1), ra);
      tile_load16(tile_g(P, cr.jb, k + 1), rb);
    }
    mfma_abt(XA, XB, acc, sgn, lower_only);
    if (!more) break;
    if (!pre) {
      chain_wait(P, factor_flag(P, cr.ra, k + 1), factor_flag(P, cr.jb, k + 1));
      tile_load16(tileA(k + 1), ra);
      tile_load16(tile_g(P, cr.jb, k + 1), rb);
    }
  }
  __syncthreads();
}

template <int TAG>
__device__ __forceinline__ void helper_accumulate(const PobtafChain& P, const ContribRange& cr, double sgn,
                                  bool lower_only, double* XA, double* XB, f64x4 (&acc)[2][2]) {
  if (cr.k0 >= cr.k1) return;
  if (P.f32) {
    f32x4 a32[2][2];
    cacc32_zero(a32);
    helper_products(P, cr, sgn, lower_only, XA, XB, a32);
    acc32_add(a32, acc, XA, KP);
  } else {
    helper_products(P, cr, sgn, lower_only, XA, XB, acc);
  }
}

// out = acc * Linv(j)^T
template <int TAG>
__device__ __forceinline__ void helper_solve(const PobtafChain& P, int j, double* XA, double* XB,
                             f64x4 (&acc)[2][2]) {
  chain_wait(P, P.cflags + 2 * j, nullptr);
  TileRegs16 rl;
  tile_load16({P.linv + (int64_t)j * CT * CT, CT, CT, CT}, rl);
  cacc_to_lds(acc, XA, KP);  // A[m][k] = acc(m, k)
  tile_store16(rl, XB);      // B[n][k] = Linv(n, k)
  __syncthreads();
  cacc_zero(acc);
  if (P.f32) {
    f32x4 a32[2][2];
    cacc32_zero(a32);
    mfma_abt(XA, XB, a32, 1.0, false);
    acc32_add(a32, acc, XA, KP);
  } else {
    mfma_abt(XA, XB, acc, 1.0, false);
  }
}

// ------------------------------------------------------------- chain work
// Columns p .. p + 15 of the factored tile S to memory by the calling wave,
// zeros above the diagonal.
__device__ __forceinline__ void chain_store_panel(const double (*S)[TT_LD], int p, const CTile& t) {
  const int lane = threadIdx.x & 63, c = p + (lane & 7) * 2;
  cdbl2 v[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = (lane >> 3) + 8 * q;
    v[q].x = c <= r ? S[r][c] : 0.0;
    v[q].y = c + 1 <= r ? S[r][c + 1] : 0.0;
  }
  double* dst = t.p + (int64_t)(lane >> 3) * t.ld + c;
#pragma unroll
  for (int q = 0; q < 8; ++q) *reinterpret_cast<cdbl2u*>(dst + (int64_t)(8 * q) * t.ld) = v[q];
}

// Rows r0 .. r0 + 15 of Ps (64 x 64, K-contiguous) <- Ps Linv^T, by the calling
// wave, in place: column block J takes K < 16 J + 16 (Linv is lower
// triangular), 40 MFMA steps on four accumulators, each operand of Ps read
// once.  ACC f64x4: FP64 MFMA; f32x4: FP32 products.
template <typename ACC>
__device__ __forceinline__ void chain_trsm_rows(double* Ps, const double (*X2)[TT_LD], int r0) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  ACC c[4];
#pragma unroll
  for (int J = 0; J < 4; ++J) c[J] = ACC{0, 0, 0, 0};
  const double* pa = Ps + (r0 + li) * TT_LD + lk;
  const double* pb = &X2[li][lk];
#pragma unroll
  for (int kk = 0; kk < CT; kk += 4) {
    const double av = pa[kk];
#pragma unroll
    for (int J = kk / 16; J < 4; ++J) c[J] = mfma_acc(av, pb[16 * J * TT_LD + kk], c[J]);
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int J = 0; J < 4; ++J)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      Ps[(r0 + acc_row(c[J], lane, r)) * TT_LD + 16 * J + acc_col(lane)] = (double)c[J][r];
}

// The ten lower 16 x 16 blocks of a 64-tile dealt to the four waves (3, 3, 2,
// 2): block i of the calling wave, i < chain_nblk().
__device__ __forceinline__ int chain_nblk(int wave) { return wave < 2 ? 3 : 2; }
__device__ __forceinline__ void chain_blk(int wave, int i, int& rb, int& cb) {
  rb = wave == 0 ? (i > 0 ? 1 : 0) : (wave == 1 ? 2 : 3);
  cb = wave == 0 ? (i == 2 ? 1 : 0) : (wave == 3 ? i + 2 : i);
}

// The calling wave's blocks of the diagonal tile t, in the accumulator layout
// of ACC; a ragged tile continues with the identity.
template <typename ACC>
__device__ __forceinline__ void chain_pd_load(const CTile& t, int wave, f64x4 (&pd)[3]) {
  const int lane = threadIdx.x & 63;
  auto each = [&](auto&& value) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (i >= chain_nblk(wave)) break;
      int rb, cb;
      chain_blk(wave, i, rb, cb);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        pd[i][r] = value(16 * rb + acc_row(ACC{}, lane, r), 16 * cb + acc_col(lane));
    }
  };
  if (t.rows == CT)
    each([&](int row, int col) { return t.p[(int64_t)row * t.ld + col]; });
  else
    each([&](int row, int col) {
      return row < t.rows && col < t.rows ? t.p[(int64_t)row * t.ld + col] : (row == col ? 1.0 : 0.0);
    });
}

// The calling wave's blocks of Sn <- pd - Ps Ps^T.
template <typename ACC>
__device__ __forceinline__ void chain_syrk(const double* Ps, const f64x4 (&pd)[3], int wave,
                                           double* Sn) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int nblk = chain_nblk(wave);
  ACC acc[3];
  const double* pa[3];
  const double* pb[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    int rb, cb;
    chain_blk(wave, i, rb, cb);
    pa[i] = Ps + (16 * rb + li) * TT_LD + lk;
    pb[i] = Ps + (16 * cb + li) * TT_LD + lk;
    acc[i] = ACC{0, 0, 0, 0};
    if constexpr (sizeof(ACC) == sizeof(f64x4)) acc[i] = pd[i];
  }
  if (nblk == 3) {
#pragma unroll
    for (int kk = 0; kk < CT; kk += 4)
#pragma unroll
      for (int i = 0; i < 3; ++i) acc[i] = mfma_acc(-pa[i][kk], pb[i][kk], acc[i]);
  } else {
#pragma unroll
    for (int kk = 0; kk < CT; kk += 4)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = mfma_acc(-pa[i][kk], pb[i][kk], acc[i]);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i >= nblk) break;
    int rb, cb;
    chain_blk(wave, i, rb, cb);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double v = (double)acc[i][r];
      if constexpr (sizeof(ACC) != sizeof(f64x4)) v += pd[i][r];
      Sn[(16 * rb + acc_row(acc[i], lane, r)) * TT_LD + 16 * cb + acc_col(lane)] = v;
    }
  }
}

// ------------------------------------------------------------- chain step
// Step g starts with D(g,g) fully updated in S and:
//   1. factors it (wave 0 factors the 16-column panels; waves 1-3 update the
//      trailing columns and form block rows 1 and 2 of Linv(g) beside them;
//      the diagonal blocks of Linv(g) come with the panels);
//   2. completes Linv(g) (block row 3), stores it and releases it: the helpers
//      wait for it first;
//   3. with PX(g) staged in Ps, L(g+1,g) = PX(g) Linv(g)^T, 16 rows per wave;
//   4. D(g+1,g+1) = PD(g+1) - L(g+1,g) L(g+1,g)^T on its lower 16 x 16
//      blocks, into the other D buffer.
// L(g+1,g) is released at the start of step g+1, whose first panel only wave
// 0 works on.  In the mixed mode the products of steps 3 and 4 round their
// operands to FP32 and accumulate in FP32; the PD(g+1) term stays FP64.
// A ragged tile (the last of a block when b % 64 != 0) runs padded with the
// identity to 64: PX comes with zeros past its rows and columns, so the
// padding stays what it is through steps 3 and 4, and only the 16-column
// panels that hold columns of the matrix are factored (chain_factor_ragged).
// Measured against a schedule of their own with ragged tile routines: n = 100,
// b = 130, a = 0 4.26 (5.22) ms, n = 8, b = 96, a = 12 248 (354) us.
// Arrows of more than one tile add helper tasks only: n = 24, b = 200, a = 70
// 1.39 ms, 3.9 ms launch per tile.
// LDS: two D buffers [64][65] (D(g,g) -> L(g,g), and D(g+1,g+1)), Xs
// [64][65] (Linv(g)), Ps [64][65] (PX(g) -> L(g+1,g), row-major =
// K-contiguous).
//
// chain_factor_ragged: L(g,g) of m < 64 columns in S, Linv(g) in X2 (the
// identity past m), L(g,g) to memory; wave 3 looks at the flags of PX(g) and
// PD(g+1) meanwhile.  Returns with every wave past the last write of X2.
template <int TAG>
__device__ __forceinline__ void chain_factor_ragged(const PobtafChain& P, double (*S2)[TT_LD],
                                                    double (*X2)[TT_LD], int m, int64_t row0,
                                                    const CTile& dt, bool sub, const int* f_px,
                                                    const int* f_pd, int* s_early) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pe = (m + PW - 1) / PW * PW;  // columns factored
  for (int idx = pe * CT + tid; idx < CT * CT; idx += CH_THREADS)
    X2[idx / CT][idx % CT] = idx / CT == idx % CT ? 1.0 : 0.0;
#pragma unroll 1
  for (int p = 0; p < pe; p += PW) {
    if (wave == 0) {
      WavePanel16<true> w;
      w.factor(S2, p, TT);
      w.finish(S2, p, &X2[p][p], TT_LD, P.info, row0);
    }
    __syncthreads();
    if (p + PW < pe) {
      lds_syrk_cols(S2, p, p + PW, pe, 0, 4);
      __syncthreads();
    }
  }
#pragma unroll 1
  for (int I = 1; I < pe / PW; ++I) {
    if (wave < I) wave_trtri_offdiag(S2, X2, &X2[PW * I][PW * I], TT_LD, I, wave);
    __syncthreads();
  }
  if (wave == 3) {
    int ok = sub ? (__hip_atomic_load(f_px, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &
                    __hip_atomic_load(f_pd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                 : 0;
    ok = __builtin_amdgcn_readfirstlane(ok);
    if (ok) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if ((tid & 63) == 0) *s_early = ok;
  }
  for (int idx = tid; idx < m * CT; idx += CH_THREADS) {
    const int r = idx / CT, c = idx % CT;
    if (c < m) dt.p[(int64_t)r * dt.ld + c] = c <= r ? S2[r][c] : 0.0;
  }
  __syncthreads();
}

template <int TAG>
__device__ __forceinline__ void chain_run(const PobtafChain& P, double* Sa, double* Sb,
                                                double* Xs, double* Ps) {
  const int tid = threadIdx.x;
  double (*X2)[TT_LD] = reinterpret_cast<double (*)[TT_LD]>(Xs);
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rs = tid >> 5, c2 = (tid & 31) * 2;
  constexpr int PUB = 64;  // wave 1, lane 0: runs the releases
  for (int idx = tid; idx < CT * TT_LD; idx += CH_THREADS) Xs[idx] = 0.0;
  {
    f64x4 acc[2][2];
    cacc_load(tile_g(P, 0, 0), acc);  // D(0,0) has no updates
    cacc_to_lds(acc, Sa, TT_LD);
    __syncthreads();
    const int m0 = cmin(CT, P.b);
    if (tid >= m0 && tid < CT) Sa[tid * TT_LD + tid] = 1.0;
  }
  __syncthreads();
  __shared__ int s_early;
  int pending = -1;  // step whose L(g+1,g) stores wait for their release
  double* S = Sa;
  double* Sn = Sb;
  for (int g = 0; g < P.NT; ++g) {
    double (*S2)[TT_LD] = reinterpret_cast<double (*)[TT_LD]>(S);
    const CTile dt = tile_g(P, g, g);
    const bool sub = g + 1 < band_end(P, g);
    const int* f_px = P.hflags + t_px(P, g);
    const int* f_pd = sub ? P.hflags + t_pd(P, g + 1) : f_px;
    if (pending >= 0 && tid == PUB) {
      // every wave waited for its L(g,g-1) stores before the barrier that
      // ended the previous step
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      wave_stores_done();
      __hip_atomic_store(P.cflags + 2 * pending + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    pending = -1;
    chain_trace(P, g, 0);
    // 1. factorization with Linv block rows 1 and 2 and the stores of
    //    finished panels beside it; PX(g) and PD(g+1) flags checked by wave 1
    //    during the last panel
    const int64_t row0 = (int64_t)(g / P.nt) * P.b + (int64_t)(g % P.nt) * CT;
    const int m = dt.rows;
    if (m == CT) lds_potrf_t<CT>(S2, X2, CT, P.info, row0, [&](int p) {
      if (p < 32) {
        if (wave == 3) chain_store_panel(S2, p, dt);
        if (p == 16 && wave == 2) wave_trtri_offdiag(S2, X2, &X2[16][16], TT_LD, 1, 0);
      } else if (wave == 1) {
        chain_store_panel(S2, 32, dt);
        // a few looks: a flag set while the panel runs saves the wait after it
        int ok = 0;
        for (int look = 0; sub && !ok && look < 3; ++look)
          ok = __builtin_amdgcn_readfirstlane(
              __hip_atomic_load(f_px, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &
              __hip_atomic_load(f_pd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (ok) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (lane == 0) s_early = ok;
      } else {
        wave_trtri_offdiag(S2, X2, &X2[32][32], TT_LD, 2, wave == 2 ? 1 : 0);
      }
    });
    else
      chain_factor_ragged<TAG>(P, S2, X2, m, row0, dt, sub, f_px, f_pd, &s_early);
    const int early = s_early;
    chain_trace(P, g, 1);
    // PX(g) and PD(g+1), if both were published during the factorization: the
    // loads land during step 2
    const CTile xt = tile_g(P, g + 1, g);
    TileRegs16 rx;
    f64x4 pd[3];
    auto load_px = [&]() {
      tile_load16(xt, rx);
      if (P.f32)
        chain_pd_load<f32x4>(tile_g(P, g + 1, g + 1), wave, pd);
      else
        chain_pd_load<f64x4>(tile_g(P, g + 1, g + 1), wave, pd);
    };
    auto stage_px = [&]() {  // pitch 65: 8-byte stores
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        Ps[(rs + 8 * q) * TT_LD + c2] = rx.v[q].x;
        Ps[(rs + 8 * q) * TT_LD + c2 + 1] = rx.v[q].y;
      }
    };
    if (early) load_px();
    // 2. Linv block row 3; the last panel of L(g,g) and Linv(g) to memory
    if (m == CT) {
      if (wave >= 1)
        wave_trtri_offdiag(S2, X2, &X2[48][48], TT_LD, 3, wave - 1);
      else
        chain_store_panel(S2, 48, dt);
      __syncthreads();
    }
    double* li_out = P.linv + (int64_t)g * CT * CT;
    {
      cdbl2 v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        v[q].x = X2[rs + 8 * q][c2];
        v[q].y = X2[rs + 8 * q][c2 + 1];
      }
      if (m < CT) {  // zeros past a ragged tile's rows and columns
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          if (rs + 8 * q >= m || c2 >= m) v[q].x = 0.0;
          if (rs + 8 * q >= m || c2 + 1 >= m) v[q].y = 0.0;
        }
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) *reinterpret_cast<cdbl2*>(li_out + (rs + 8 * q) * CT + c2) = v[q];
    }
    if (!sub) {  // last diagonal tile of the matrix
      chain_publish(P.cflags + 2 * g);
      continue;
    }
    if (early) stage_px();
    wave_stores_done();
    __syncthreads();
    if (tid == PUB) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      wave_stores_done();
      __hip_atomic_store(P.cflags + 2 * g, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!early) {
      wave_wait(P, f_px, f_pd);
      load_px();
      stage_px();
      __syncthreads();
    }
    chain_trace(P, g, 2);
    // 3. L(g+1,g), wave w: rows 16w .. 16w + 15
    if (P.f32)
      chain_trsm_rows<f32x4>(Ps, X2, 16 * wave);
    else
      chain_trsm_rows<f64x4>(Ps, X2, 16 * wave);
    __syncthreads();  // L(g+1,g) complete in Ps
    chain_trace(P, g, 3);
    lds_tile_store(Ps, TT_LD, xt);
    pending = g;
    // 4. D(g+1,g+1) into Sn
    if (P.f32)
      chain_syrk<f32x4>(Ps, pd, wave, Sn);
    else
      chain_syrk<f64x4>(Ps, pd, wave, Sn);
    wave_stores_done();  // L(g+1,g): released at the start of step g+1
    __syncthreads();
    chain_trace(P, g, 5);
    double* t = S;
    S = Sn;
    Sn = t;
  }
  if (pending >= 0 && tid == PUB) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    wave_stores_done();
    __hip_atomic_store(P.cflags + 2 * pending + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---------------------------------------------------------------- kernel
// One helper task (already claimed) of matrix P.
template <int TAG>
__device__ __forceinline__ void chain_helper_task(const PobtafChain& P, int task, double* lds) {
  const int tid = threadIdx.x;
  double* XA = lds;
  double* XB = lds + CT * KP;
  int r, j;
  const int kind = chain_decode(P, task, r, j);
  if (kind == HK_NOOP) return;  // nobody waits on an empty slot

  f64x4 acc[2][2];
  if (kind == HK_TIP) {
    cacc_load({P.T, P.a, P.a, P.a}, acc);
    // four products a round: one round trip for their loads
    for (int i0 = 0; i0 < P.n; i0 += 4) {
      f64x4 pi[4][2][2];
      if (tid == 0) {
        long long spins = 0;
        for (int i = i0; i < i0 + 4 && i < P.n; ++i)
          if (!chain_poll(P, P.hflags + t_tippc(P, i), spins)) {
            __hip_atomic_store(P.info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + u < P.n) cacc_load({P.tipp + (int64_t)(i0 + u) * P.a * P.a, P.a, P.a, P.a}, pi[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + u < P.n) {
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[x][y] -= pi[u][x][y];
        }
    }
    double (*S2)[TT_LD] = reinterpret_cast<double (*)[TT_LD]>(lds);
    cacc_to_lds(acc, lds, TT_LD);
    __syncthreads();
    double (*X2)[TT_LD] = reinterpret_cast<double (*)[TT_LD]>(lds + CT * TT_LD);
    lds_potrf(S2, X2, P.a, P.info, (int64_t)P.n * P.b);
    for (int idx = tid; idx < P.a * P.a; idx += CH_THREADS) {
      const int rr = idx / P.a, cc = idx % P.a;
      P.T[idx] = (cc <= rr) ? S2[rr][cc] : 0.0;
    }
    if (P.tip_inv) {
      double (*W2)[WS_LD] = reinterpret_cast<double (*)[WS_LD]>(lds + 2 * CT * TT_LD);
      __syncthreads();
      lds_trtri(S2, X2, W2, P.a);
      for (int idx = tid; idx < CT * CT; idx += CH_THREADS) {
        const int rr = idx / CT, cc = idx % CT;
        P.tip_inv[idx] = (rr < P.a && cc <= rr) ? X2[rr][cc] : 0.0;
      }
    }
    chain_publish(P.hflags + task);
    return;
  }
  if (kind == HK_TIPP) {
    const int i = j;
    cacc_zero(acc);
    for (int c = 0; c < P.nt; ++c) {
      const int k = i * P.nt + c;
      chain_wait(P, P.hflags + t_arr(P, k, 0), nullptr);
      TileRegs16 x;
      tile_load16(tile_arrow(P, k, 0), x);
      __syncthreads();
      tile_store16(x, XA);
      __syncthreads();
      mfma_abt(XA, XA, acc, 1.0, true);
    }
    cacc_store({P.tipp + (int64_t)i * P.a * P.a, P.a, P.a, P.a}, acc);  // FP64 (tip path)
    chain_publish(P.hflags + task);
    return;
  }
  CTile out;
  if (kind == HK_TRSM)
    out = tile_g(P, r, j);
  else if (kind == HK_ARR)
    out = tile_arrow(P, j, r);
  else if (kind == HK_PX)
    out = tile_g(P, j + 1, j);
  else
    out = tile_g(P, j, j);  // PD
  cacc_load(out, acc);
  const ContribRange cr = chain_contribs(P, kind, r, j);
  helper_accumulate<TAG>(P, cr, -1.0, kind == HK_PD, XA, XB, acc);
  if (kind == HK_TRSM || kind == HK_ARR) helper_solve<TAG>(P, j, XA, XB, acc);
  __syncthreads();  // the last product is done with XA
  cacc_to_lds(acc, XA, KP);
  __syncthreads();
  lds_tile_store(XA, KP, out);
  chain_publish(P.hflags + task);
  if (kind == HK_PX) chain_trace(P, j, 6);
  if (kind == HK_TRSM && r == j + 2) chain_trace(P, j, 7);
  // The strict-upper mirror of a lower D-block tile is zero in the factor.
  // No task reads it, so it is cleared after the publish, off the path of
  // the tasks waiting for this one.
  if (kind == HK_TRSM && r / P.nt == j / P.nt) tile_zero(tile_mirror(P, r, j));
  if (kind == HK_PX && (j + 1) / P.nt == j / P.nt) tile_zero(tile_mirror(P, j + 1, j));
}

// LDS: the helper plan (XA, XB) or the chain's (two D buffers, Xs, Ps),
// whichever is larger.
constexpr int CH_LDS_HELPER = 2 * CT * KP + CT * WS_LD;
constexpr int CH_LDS_CHAIN = 4 * CT * TT_LD;
constexpr int CH_LDS = CH_LDS_HELPER > CH_LDS_CHAIN ? CH_LDS_HELPER : CH_LDS_CHAIN;

__global__ void __launch_bounds__(CH_THREADS) pobtaf_chain_kernel(PobtafChain P) {
  __shared__ __attribute__((aligned(16))) double lds[CH_LDS];
  __shared__ int s_task;
  const int tid = threadIdx.x;
  if (tid == 0) s_task = atomicAdd(P.claim, 1);
  __syncthreads();
  const bool is_chain = (s_task == 0);
  __syncthreads();
  if (is_chain) {
    // the chain runs latency-bound code: keep helpers off its CU
    if (tid == 0)
      __hip_atomic_store(P.chain_cu, 1 + hw_cu_key(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    chain_run<0>(P, lds, lds + CT * TT_LD, lds + 2 * CT * TT_LD, lds + 3 * CT * TT_LD);
    return;
  }
  const int my_cu = 1 + hw_cu_key();
  for (;;) {
    if (tid == 0) {
      const int ccu = __hip_atomic_load(P.chain_cu, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_task = (ccu == my_cu) ? P.ntasks : atomicAdd(P.counter, 1);
    }
    __syncthreads();
    const int task = s_task;
    __syncthreads();
    if (task >= P.ntasks) return;
    chain_helper_task<0>(P, task, lds);
  }
}

// Many independent matrices in one persistent launch (batched plans).  The
// first nmat claims of *gclaim become the chains of matrices 0..nmat-1; every
// other workgroup serves one matrix's helper queue in order until it is
// drained, then the next one's, and leaves when a full round finds every queue
// drained.  It starts at its home (helper_home; nres: workgroups resident at
// once).  With fewer helpers than matrices they go round after every task, so
// that no chain waits for others to end.  Going round the matrices after every task instead left the longest
// chain waiting for helpers: 24.7 ms for 64 systems of up to 1024 diagonal
// tiles.  cu_busy (4096 ints, zero on entry) marks the CUs that run a chain;
// helpers there leave at once.
__global__ void __launch_bounds__(CH_THREADS) pobtaf_chain_multi_kernel(const PobtafChain* Ps,
                                                                        int nmat, int nres,
                                                                        int* gclaim, int* cu_busy) {
  __shared__ __attribute__((aligned(16))) double lds[CH_LDS];
  __shared__ int s_task;
  const int tid = threadIdx.x;
  if (tid == 0) s_task = atomicAdd(gclaim, 1);
  __syncthreads();
  const int first = s_task;
  __syncthreads();
  const int my_key = hw_cu_key() & 4095;
  if (first < nmat) {
    if (tid == 0) __hip_atomic_store(cu_busy + my_key, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const PobtafChain& P = Ps[first];
    chain_run<1>(P, lds, lds + CT * TT_LD, lds + 2 * CT * TT_LD, lds + 3 * CT * TT_LD);
    return;
  }
  if (tid == 0)
    s_task = helper_home(first - nmat, nres - nmat, nmat, [&](int i) {
      const double nt = Ps[i].nt;  // products of a step's tasks, and a part per task
      return Ps[i].NT * (3.0 + nt * (5.0 + 3.0 * nt));
    });
  __syncthreads();
  int m = s_task;
  __syncthreads();
  const bool stay = nres - nmat >= nmat;
  int drained = 0;  // consecutive matrices found without tasks
  while (drained < nmat) {
    const PobtafChain& P = Ps[m];
    if (tid == 0) {
      const int busy = __hip_atomic_load(cu_busy + my_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_task = busy ? -1 : atomicAdd(P.counter, 1);
    }
    __syncthreads();
    const int task = s_task;
    __syncthreads();
    if (task < 0) return;
    if (task >= P.ntasks) {
      ++drained;
      m = (m + 1 == nmat) ? 0 : m + 1;
    } else {
      drained = 0;
      chain_helper_task<1>(P, task, lds);
      if (!stay) m = (m + 1 == nmat) ? 0 : m + 1;
    }
  }
}

}  // namespace rocbta
