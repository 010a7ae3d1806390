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
// Memory ordering: the helpers' TRSM, ARR, PX and PD tiles and the chain's
// Linv(g) are written through (agent-scope stores), each wave adding its share
// to the flag once its own stores are complete: no barrier and no cache
// write-back between a tile and its readers.  The chain's L(g+1,g) uses plain
// stores, whose issue does not hold a wave up, and one release by wave 3 at the
// start of the next step; TIPP and TIP are published behind a barrier and one
// release (chain_publish).  A tile is ready when its flag holds CH_READY;
// waiters poll relaxed and issue one agent-scope acquire.
#pragma once
#include "common.hpp"
#include "tile_f64.hpp"

namespace rocbta {

constexpr int CT = 64;          // tile size
constexpr int CH_THREADS = 256;
constexpr int KP = CT + 2;      // pitch of K-contiguous LDS tiles (doubles)
constexpr int CH_READY = 12;    // flag of a published tile

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
//   0 step start, 1 factorization done, 2 Linv(g) complete, PX(g)/PD(g+1)
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
__device__ __forceinline__ bool chain_ready(const int* f) {
  return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= CH_READY;
}
__device__ __forceinline__ bool chain_poll(const PobtafChain& P, const int* f, long long& spins) {
  while (!chain_ready(f)) {
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
__device__ __forceinline__ void chain_publish(int* f) {
  wave_stores_done();
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    wave_stores_done();
    __hip_atomic_store(f, CH_READY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The calling wave's share of a tile that several waves write through.
__device__ __forceinline__ void chain_wave_done(int* f, int share) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // also keeps the stores above it
  if ((threadIdx.x & 63) == 0)
    __hip_atomic_fetch_add(f, share, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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

// 16 bytes written through to where every XCD reads them (agent scope).  The
// wait state keeps the data registers until the store has taken them.
__device__ __forceinline__ void store_through(double* p, const cdbl2& v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 0" : : "v"(p), "v"(v) : "memory");
}

// Rows r0 .. r0 + NR - 1 (NR even) of the LDS tile X to tile t by the calling
// wave, written through; zeros past row and column mc of t (mc = 64: none).
template <int NR>
__device__ __forceinline__ void chain_store_rows(const double* X, int pitch, int r0, const CTile& t,
                                                 int mc = CT) {
  const int lane = fresh_lane(), rs = r0 + (lane >> 5), c = 2 * (lane & 31);
  cdbl2 v[NR / 2];
#pragma unroll
  for (int q = 0; q < NR / 2; ++q) {
    const double* x = X + (rs + 2 * q) * pitch + c;
    v[q].x = x[0];
    v[q].y = x[1];
  }
  if (mc < CT) {
#pragma unroll
    for (int q = 0; q < NR / 2; ++q) {
      if (rs + 2 * q >= mc || c >= mc) v[q].x = 0.0;
      if (rs + 2 * q >= mc || c + 1 >= mc) v[q].y = 0.0;
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // all reads before the first store
  double* dst = t.p + (int64_t)rs * t.ld + c;
  if (t.rows == CT && t.cols == CT) {
#pragma unroll
    for (int q = 0; q < NR / 2; ++q) store_through(dst + (int64_t)(2 * q) * t.ld, v[q]);
  } else {
#pragma unroll
    for (int q = 0; q < NR / 2; ++q) {
      double* d = dst + (int64_t)(2 * q) * t.ld;
      if (rs + 2 * q >= t.rows) continue;
      if (c < t.cols) __hip_atomic_store(d, v[q].x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (c + 1 < t.cols) __hip_atomic_store(d + 1, v[q].y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
// Rows r0 .. r0 + 15 of Ps (64 x 64, K-contiguous, pitch LD) <- Ps Linv^T, by the calling
// wave, in place: column block J takes K < 16 J + 16 (Linv is lower
// triangular), 40 MFMA steps on four accumulators, each operand of Ps read
// once.  ACC f64x4: FP64 MFMA; f32x4: FP32 products.
template <typename ACC, int LD>
__device__ __forceinline__ void chain_trsm_rows(double* Ps, const double* Linv, int r0) {
  const int lane = fresh_lane(), li = lane & 15, lk = lane >> 4;
  ACC c[4];
#pragma unroll
  for (int J = 0; J < 4; ++J) c[J] = ACC{0, 0, 0, 0};
  const double* pa = Ps + (r0 + li) * LD + lk;
  const double* pb = Linv + li * LD + lk;
  // operands of 16 k at a time, read while the previous 16 are multiplied
  double a[2][4], b[2][4][4];
  auto fetch = [&](int buf, int K) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a[buf][u] = pa[16 * K + 4 * u];
#pragma unroll
      for (int J = 0; J < 4; ++J)
        if (J >= K) b[buf][u][J] = pb[16 * J * LD + 16 * K + 4 * u];
    }
  };
  fetch(0, 0);
#pragma unroll
  for (int K = 0; K < 4; ++K) {
    if (K < 3) fetch((K + 1) & 1, K + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int J = 0; J < 4; ++J)
        if (J >= K) c[J] = mfma_acc(a[K & 1][u], b[K & 1][u][J], c[J]);
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int J = 0; J < 4; ++J)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      Ps[(r0 + acc_row(c[J], lane, r)) * LD + 16 * J + acc_col(lane)] = (double)c[J][r];
}

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
  // each operand is loaded as soon as it is there
  auto wait_load = [&](int k) {
    chain_wait(P, factor_flag(P, cr.ra, k), nullptr);
    tile_load16(tileA(k), ra);
    if (!(cr.ra == cr.jb)) chain_wait(P, factor_flag(P, cr.jb, k), nullptr);
    tile_load16(tile_g(P, cr.jb, k), rb);
  };
  wait_load(cr.k0);
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
      if (more && chain_ready(factor_flag(P, cr.ra, k + 1)) && chain_ready(factor_flag(P, cr.jb, k + 1))) {
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
      wait_load(k + 1);
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

// XA <- acc * Linv(j)^T, rows 16w .. 16w + 15 by wave w (complete for that wave).
__device__ __forceinline__ void helper_solve(const PobtafChain& P, int j, double* XA, double* XB,
                                             const f64x4 (&acc)[2][2]) {
  chain_wait(P, P.cflags + 2 * j, nullptr);
  TileRegs16 rl;
  tile_load16({P.linv + (int64_t)j * CT * CT, CT, CT, CT}, rl);
  cacc_to_lds(acc, XA, KP);  // A[m][k] = acc(m, k)
  tile_store16(rl, XB);      // B[n][k] = Linv(n, k)
  __syncthreads();
  if (P.f32)
    chain_trsm_rows<f32x4, KP>(XA, XB, 16 * wave_id());
  else
    chain_trsm_rows<f64x4, KP>(XA, XB, 16 * wave_id());
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// ------------------------------------------------------------- chain work
// Rows r0 .. r0 + NR - 1 (NR even) of the LDS tile X to tile t by the calling
// wave; LOWER: zeros above the diagonal (t full).
template <int NR, bool LOWER>
__device__ __forceinline__ void chain_store_plain(const double* X, int r0, const CTile& t) {
  const int lane = fresh_lane(), rs = r0 + (lane >> 5), c = 2 * (lane & 31);
  cdbl2 v[NR / 2];
#pragma unroll
  for (int q = 0; q < NR / 2; ++q) {
    const double* x = X + (rs + 2 * q) * TT_LD + c;
    v[q].x = x[0];
    v[q].y = x[1];
  }
  if (LOWER) {
#pragma unroll
    for (int q = 0; q < NR / 2; ++q) {
      if (c > rs + 2 * q) v[q].x = 0.0;
      if (c + 1 > rs + 2 * q) v[q].y = 0.0;
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // all reads before the first store
  double* dst = t.p + (int64_t)rs * t.ld + c;
  if (LOWER || (t.rows == CT && t.cols == CT)) {
#pragma unroll
    for (int q = 0; q < NR / 2; ++q) *reinterpret_cast<cdbl2u*>(dst + (int64_t)(2 * q) * t.ld) = v[q];
  } else {
#pragma unroll
    for (int q = 0; q < NR / 2; ++q) {
      double* d = dst + (int64_t)(2 * q) * t.ld;
      if (rs + 2 * q < t.rows && c < t.cols) d[0] = v[q].x;
      if (rs + 2 * q < t.rows && c + 1 < t.cols) d[1] = v[q].y;
    }
  }
}

// N 16 x 16 blocks (I[i], J[i]) of X2 to the Linv tile at p, written through.
template <int N>
__device__ __forceinline__ void chain_store_blocks(const double (*X2)[TT_LD], const int (&I)[N],
                                                   const int (&J)[N], double* p) {
  const int lane = fresh_lane(), row = lane >> 3, col = 2 * (lane & 7);
  cdbl2 v[N][2];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const double* x = &X2[16 * I[i] + 8 * h + row][16 * J[i] + col];
      v[i][h].x = x[0];
      v[i][h].y = x[1];
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      store_through(p + (16 * I[i] + 8 * h + row) * CT + 16 * J[i] + col, v[i][h]);
}

// A whole tile in one wave: lane l holds rows 2q + l / 32, columns 2 (l % 32)
// and the next.  Ragged tiles continue with zeros, or with the identity.
struct WaveTile {
  cdbl2 v[32];
};
__device__ __forceinline__ void wave_tile_load(const CTile& t, bool ident, WaveTile& x) {
  const int lane = fresh_lane(), r0 = lane >> 5, c = (lane & 31) * 2;
  const double* src = t.p + (int64_t)r0 * t.ld + c;
  if (t.rows == CT && t.cols == CT) {
#pragma unroll
    for (int q = 0; q < 32; ++q) x.v[q] = *reinterpret_cast<const cdbl2u*>(src + (int64_t)(2 * q) * t.ld);
  } else {
#pragma unroll
    for (int q = 0; q < 32; ++q) {
      const int r = 2 * q + r0;
      const bool in = r < t.rows;
      x.v[q].x = in && c < t.cols ? src[(int64_t)(2 * q) * t.ld] : (ident && r == c ? 1.0 : 0.0);
      x.v[q].y = in && c + 1 < t.cols ? src[(int64_t)(2 * q) * t.ld + 1] : (ident && r == c + 1 ? 1.0 : 0.0);
    }
  }
}
__device__ __forceinline__ void wave_tile_store(const WaveTile& x, double* X) {
  const int lane = fresh_lane(), r0 = lane >> 5, c = (lane & 31) * 2;
#pragma unroll
  for (int q = 0; q < 32; ++q) {
    X[(2 * q + r0) * TT_LD + c] = x.v[q].x;
    X[(2 * q + r0) * TT_LD + c + 1] = x.v[q].y;
  }
}

// N 16 x 16 blocks of Sn -= Ps Ps^T by the calling wave: rows rb[i], columns cb[i].
template <typename ACC, int N>
__device__ __forceinline__ void chain_syrk(const double* Ps, double* Sn, const int (&rb)[N],
                                           const int (&cb)[N]) {
  const int lane = fresh_lane(), li = lane & 15, lk = lane >> 4;
  constexpr bool wide = sizeof(ACC) == sizeof(f64x4);
  ACC acc[N];
  double* c[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    c[i] = Sn + (16 * rb[i] + acc_row(ACC{}, lane, 0)) * TT_LD + 16 * cb[i] + acc_col(lane);
    acc[i] = ACC{0, 0, 0, 0};
    if constexpr (wide) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][r] = c[i][4 * r * TT_LD];
    }
  }
  double a[2][4][N], b[2][4][N];
  auto fetch = [&](int buf, int K) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        a[buf][u][i] = Ps[(16 * rb[i] + li) * TT_LD + 16 * K + 4 * u + lk];
        b[buf][u][i] = Ps[(16 * cb[i] + li) * TT_LD + 16 * K + 4 * u + lk];
      }
  };
  fetch(0, 0);
#pragma unroll
  for (int K = 0; K < 4; ++K) {
    if (K < 3) fetch((K + 1) & 1, K + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < N; ++i) acc[i] = mfma_acc(-a[K & 1][u][i], b[K & 1][u][i], acc[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (wide)
        c[i][4 * r * TT_LD] = acc[i][r];
      else
        c[i][r * TT_LD] += (double)acc[i][r];
    }
}

// ------------------------------------------------------------- chain step
// Step g starts with the first 16 columns of D(g,g) updated in S, and:
//   1. factors it.  Wave 0 factors the 16-column panels.  Beside them waves 1-3
//      finish the update of the other columns by L(g,g-1) and apply the panels
//      to them; wave 3 forms block rows 1 and 2 of Linv(g) (its diagonal
//      blocks come with the panels) and the products of row 3; waves 1 and 2
//      store L(g-1,g-1) and, during the last panel, look whether PX(g) and
//      PD(g+1) are published and load them if so;
//   2. wave 3 completes Linv(g) while waves 1 and 2 wait for PX(g) and PD(g+1)
//      if need be and put them in Ps and the other D buffer;
//   3. L(g+1,g) = PX(g) Linv(g)^T, 16 rows per wave; Linv(g) is flagged after
//      it, or before it if PX(g) was late: its stores have landed by then;
//   4. the first 16 columns of D(g+1,g+1) = PD(g+1) - L(g+1,g) L(g+1,g)^T;
//      L(g+1,g), stored meanwhile, is released beside the next first panel.
// On the path are the four panels (8 us), 12 MFMA steps of the block row, 40 of
// the solve, 16 of the update, and four barriers.  Stores and flag reads stay
// off it: a wave that waits for either holds the next barrier up, so wave 0
// has none, and no store precedes a look in the same phase.  In the mixed mode
// the products of steps 3 and 4 round their operands to FP32 and accumulate in
// FP32; the PD(g+1) term stays FP64.
// Measured, median step at b = 64 / 256 / 1024: 12.1 / 12.7 / 13.9 us; with
// whole update and release between the steps 14.2 / 14.2 / 15.1 us.  From b = 256
// on PX(g) arrives about when the panels end: the helpers' path from Linv(g)
// over L(g+2,g) to PX(g+1) is as long as the chain's.
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
// chain_factor_ragged: L(g,g) of m < 64 columns in S and in memory, Linv(g) in
// X2 (the identity past m).  start() and rest() run on waves 1-3 and
// store_prev() on waves 1 and 2 beside the first panel, look() there beside the
// last.  Ends with a barrier.
template <typename START, typename REST, typename PREV, typename LOOK>
__device__ __forceinline__ void chain_factor_ragged(double (*S2)[TT_LD], double (*X2)[TT_LD], int m,
                                                    int* info, int64_t row0, const CTile& dt,
                                                    const START& start, const REST& rest,
                                                    const PREV& store_prev, const LOOK& look) {
  const int tid = threadIdx.x, wave = wave_id();
  const int pe = (m + PW - 1) / PW * PW;  // columns factored
  for (int idx = pe * CT + tid; idx < CT * CT; idx += CH_THREADS)
    X2[idx / CT][idx % CT] = idx / CT == idx % CT ? 1.0 : 0.0;
#pragma unroll 1
  for (int p = 0; p < pe; p += PW) {
    if (wave == 0) {
      WavePanel16<true> w;
      w.factor(S2, p, TT);
      w.finish(S2, p, &X2[p][p], TT_LD, info, row0);
    } else {
      if (p == 0) {
        start();
        rest();
        if (wave < 3) store_prev();
      }
      if (p + PW >= pe && wave < 3) look(3);
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
  for (int idx = tid; idx < m * CT; idx += CH_THREADS) {
    const int r = idx / CT, c = idx % CT;
    if (c < m) dt.p[(int64_t)r * dt.ld + c] = c <= r ? S2[r][c] : 0.0;
  }
}

template <int TAG>
__device__ __forceinline__ void chain_run(const PobtafChain& P, double* Sa, double* Sb, double* Xs,
                                          double* Ps) {
  const int tid = threadIdx.x;
  double (*X2)[TT_LD] = reinterpret_cast<double (*)[TT_LD]>(Xs);
  const int lane = tid & 63, wave = wave_id();
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
  __shared__ int s_have[2];
  bool pending = false;  // L(g,g-1) is in Ps: update, store and flag open
  double* S = Sa;
  double* Sn = Sb;
  for (int g = 0; g < P.NT; ++g) {
    double (*S2)[TT_LD] = reinterpret_cast<double (*)[TT_LD]>(S);
    const CTile dt = tile_g(P, g, g);
    const int m = dt.rows;
    const bool sub = g + 1 < band_end(P, g);
    int* const f_linv = P.cflags + 2 * g;
    double* const linv = P.linv + (int64_t)g * CT * CT;
    chain_trace(P, g, 0);
    // 1. factorization
    WaveTile wt;        // waves 1, 2: PX(g), PD(g+1)
    bool have = false;
    const int* const f_tile = !sub ? nullptr : P.hflags + (wave == 1 ? t_px(P, g) : t_pd(P, g + 1));
    auto load_tile = [&]() { wave_tile_load(tile_g(P, g + 1, g + (wave - 1)), wave == 2, wt); };
    auto syrk = [&](double* X, int rb, int cb) {
      const int r[1] = {rb}, c[1] = {cb};
      if (P.f32)
        chain_syrk<f32x4, 1>(Ps, X, r, c);
      else
        chain_syrk<f64x4, 1>(Ps, X, r, c);
    };
    auto start = [&]() {
      if (!pending) return;
      if (wave == 3) {  // every wave has waited for its rows of L(g,g-1)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        chain_wave_done(P.cflags + 2 * g - 1, CH_READY);
      }
      syrk(S, wave, 1);
    };
    // blocks (2,2), (3,2), (3,3): after the update of the same blocks by panel 0,
    // which the same waves have
    auto rest = [&]() {
      if (pending) syrk(S, wave == 1 ? 2 : 3, wave == 3 ? 3 : 2);
    };
    // waves 1, 2: L(g-1,g-1), still in the other D buffer
    auto store_prev = [&]() {
      if (!pending) return;
      const CTile pt = tile_g(P, g - 1, g - 1);
      if (pt.rows == CT) chain_store_plain<32, true>(Sn, 32 * (wave - 1), pt);
    };
    WaveTrtriRow<3> row3;  // wave 3
    auto look = [&](int looks) {
      // a few looks: a flag set while the panel runs saves the wait after it
      const bool had = have;
      for (int k = 0; sub && !have && k < looks; ++k)
        have = __builtin_amdgcn_readfirstlane((int)chain_ready(f_tile)) != 0;
      if (have && !had) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        load_tile();
      }
      if (lane == 0) s_have[wave - 1] = have;
    };
    const int64_t row0 = (int64_t)(g / P.nt) * P.b + (int64_t)(g % P.nt) * CT;
    if (m == CT) {
      lds_potrf_t<CT>(S2, X2, CT, P.info, row0, [&](int p) {
        if (p < 0) {
          start();
        } else if (p == 0) {
          rest();
        } else if (p == 16) {
          if (wave < 3) {
            store_prev();
          } else {
            WaveTrtriRow<1> row1;
            row1.products(S2, X2);
            row1.finish(X2);
            const int I[3] = {0, 1, 1}, J[3] = {0, 0, 1};
            chain_store_blocks<3>(X2, I, J, linv);
          }
        } else {
          if (wave < 3) {
            look(3);
          } else {
            WaveTrtriRow<2> row2;
            row2.products(S2, X2);
            row2.finish(X2);
            row3.products(S2, X2);
            const int I[3] = {2, 2, 2}, J[3] = {0, 1, 2};
            chain_store_blocks<3>(X2, I, J, linv);
          }
        }
      });
    } else {
      chain_factor_ragged(S2, X2, m, P.info, row0, dt, start, rest, store_prev, look);
    }
    pending = sub;
    chain_trace(P, g, 1);
    // 2. Linv(g) complete, PX(g) in Ps, PD(g+1) in Sn
    if (m < CT) {
      chain_store_rows<16>(Xs, TT_LD, 16 * wave, {linv, CT, CT, CT}, m);
    } else if (wave == 3) {
      row3.finish(X2);
      const int I[4] = {3, 3, 3, 3}, J[4] = {0, 1, 2, 3};
      chain_store_blocks<4>(X2, I, J, linv);
    }
    // Linv(g) is stored by wave 3, a ragged tile's by all waves
    const bool fetch = wave == 1 || wave == 2, stores = m < CT || wave == 3;
    const int share = m < CT ? CH_READY / 4 : CH_READY;
    const bool wait = !sub || fetch || !(s_have[0] && s_have[1]);
    if (stores && wait) chain_wave_done(f_linv, share);
    if (!sub) {  // last diagonal tile of the matrix
      if (m == CT && wave < 2) chain_store_plain<32, true>(S, 32 * wave, dt);
      continue;
    }
    if (fetch) {
      if (!have) {
        wave_wait(P, f_tile, nullptr);
        load_tile();
      }
      wave_tile_store(wt, wave == 1 ? Ps : Sn);
    }
    __syncthreads();
    chain_trace(P, g, 2);
    // 3. L(g+1,g), wave w: rows 16w .. 16w + 15
    if (P.f32)
      chain_trsm_rows<f32x4, TT_LD>(Ps, Xs, 16 * wave);
    else
      chain_trsm_rows<f64x4, TT_LD>(Ps, Xs, 16 * wave);
    if (stores && !wait) chain_wave_done(f_linv, share);
    chain_store_plain<16, false>(Ps, 16 * wave, tile_g(P, g + 1, g));
    __syncthreads();  // L(g+1,g) complete in Ps
    chain_trace(P, g, 3);
    // 4. the first 16 columns of D(g+1,g+1)
    syrk(Sn, wave, 0);
    wave_stores_done();  // L(g+1,g): released at the start of step g+1
    __syncthreads();
    chain_trace(P, g, 5);
    double* t = S;
    S = Sn;
    Sn = t;
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
  if (kind == HK_TRSM || kind == HK_ARR) {
    helper_solve(P, j, XA, XB, acc);
  } else {
    __syncthreads();  // the last product is done with XA
    cacc_to_lds(acc, XA, KP);
    __syncthreads();
  }
  chain_store_rows<16>(XA, KP, 16 * wave_id(), out);
  chain_wave_done(P.hflags + task, CH_READY / 4);
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
