// FP64 MFMA products for the quaternion panel updates and the divide & conquer.
//
// Quaternion GEMM as one real GEMM: with q = (a, b) stored as the 4-vector
// (Re a, Im a, Re b, Im b), the product q p is L(q) p with
//
//   L(q) = [ a_r  -a_i  -b_r  -b_i ]
//          [ a_i   a_r   b_i  -b_r ]
//          [ b_r  -b_i   a_r   a_i ]
//          [ b_i   b_r  -a_i   a_r ]      L(q)[r][k] = sign[r][k] * q[r ^ k].
//
// So C (m x n quaternions) += A B is the real product of L(A) (4m x 4k) with
// B viewed as a 4k x n real matrix, and each v_mfma_f64_16x16x4_f64 consumes
// 4 quaternion rows x 1 quaternion k of A (expanded on the fly from LDS) and
// 1 k x 16 quaternion columns of B.  Register layout of that instruction
// (pinned by zq_selftest_mfma): A[i][k] is in lane i + 16k, B[k][j] in lane
// j + 16k, and accumulator register r of lane l holds D[4r + l/16][l%16].
// Real row 4r + g is taken to be component r of quaternion row g, so each
// lane's four accumulators are one whole quaternion of C.  No flops are spent
// on zeros: 32 real flops per quaternion multiply-add, the count the
// roofline uses.
//
// These kernels replace the complex zgemm3m_ calls of the reference's panel
// update and Q accumulation (blocked.cc:416-544) and back-transform
// (zquatev.cc:86-90).
#include "zq_internal.h"
#include <climits>
#include <algorithm>

namespace zq {

typedef double d4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Tiles of TBM x TBN quaternions per workgroup (2 x 2 waves), K staged GBK
// quaternions at a time through double-buffered LDS.  The next stage's operands
// are fetched into registers before the current stage's MFMAs, so global
// latency hides behind the wave's own work, and one barrier per stage suffices
// (a buffer is rewritten only after the barrier that follows its last read).
// The conjugate-transpose flags are template parameters (branch-free address
// math); the sign of the L(A) expansion is applied by flipping the sign bit.
// The tile shape changes no result: an element's K-sum is one wave's
// accumulator in the same order in every shape.
//   64 x 64, GBK 8    the most reuse per fetch, for launches of very many tiles;
//                     waves of 16 x 64 read 8 fragments per 16 MFMAs where 32 x 32
//                     ones read 10 (4096 x 4096 x 1024 66.3 -> 67.3 TFLOP/s, and
//                     65.5 before the loads became branch-free, below);
//   32 x 64, GBK 8    twice the workgroups (balance, registers);
//   32 x 32, GBK 8    the same for lower-triangle products, whose K is a panel's
//                     two widths: less of the tiles above the diagonal, and four
//                     workgroups per CU (97 registers, 33 KB) to cover the
//                     reads of C.  2n = 8192 solve 144.9 -> 144.3 ms, 4096 31.93 ->
//                     31.78, batch of 512 72.6 -> 71.9; other products lose by the
//                     extra operand traffic (batch 72.0 -> 72.9);
//   16 x 32, GBK 16   for launches that leave CUs idle otherwise: a wave's time
//                     is K x (its 16 x 16 x 4 products) x 64 cycles whatever
//                     the other CUs do -- 14 us for 32 x 64 at K = 64, a
//                     quarter of that here -- and its shorter stages (1024
//                     cycles at GBK 8) would wait for the next fetch, hence 16.
//                     C is fetched before the K loop.
// ---------------------------------------------------------------------------
template <int TBM_, int TBN_, int GBK_, int WM_>
struct QTile {
  static constexpr int TBM = TBM_, TBN = TBN_, GBK = GBK_, WM = WM_;   // WM of the 4 waves along the rows
  // LDS layouts (doubles).  A: [k][row][component], B: [k][component][column],
  // each k slice padded by 2 doubles, so that fragment reads (16 consecutive
  // doubles per component group) and the stage writes of either operand
  // orientation fall in distinct banks.
  static constexpr int ASK = TBM * 4 + 2, BSK = TBN * 4 + 2;
  static constexpr bool PREC = TBM == 16;   // C fetched before the K loop
};
using Tile64 = QTile<64, 64, 8, 4>;
using Tile32 = QTile<32, 64, 8, 2>;
using Tile32L = QTile<32, 32, 8, 2>;
using Tile16 = QTile<16, 32, 16, 2>;

// Operand elements as stored, loaded without a branch at a clamped index (row
// or column i of the output, 0 <= i < m; k of the sum, within the range): a
// load in a branch is followed by a wait for it, before the current stage's
// MFMAs could start (128 x 4096 x 4096 with A transposed 53.2 -> 55.4
// TFLOP/s, 2n = 8192 solve 147.1 -> 146.1 ms).  What is out of range or masked becomes zero, and a CT operand is
// conjugated, when the stage is stashed in LDS, after those MFMAs.  A and B
// are indexed alike: storage element (i, k), for A conj-transposed and plain B (k, i).
template <bool KROW>
__device__ __forceinline__ quat ld_op(const QOperand& A, int i, int k) {
  const bool second = k >= A.ksplit;
  const quat* p = second ? A.p1 : A.p0;
  const int ld = second ? A.ld1 : A.ld0, kk = second ? k - A.ksplit : k;
  return qload_g(p + (KROW ? kk : i) + (size_t)(KROW ? i : kk) * ld);
}
// Whether that element counts: storage (r, c) is used only where r > c + mask_off.
template <bool KROW>
__device__ __forceinline__ bool op_on(const QOperand& A, int i, int k) {
  const int kk = k >= A.ksplit ? k - A.ksplit : k;
  return KROW ? kk > i + A.mask_off : i > kk + A.mask_off;
}
__device__ __forceinline__ quat qselect(bool on, const quat& v) {
  return quat{on ? v.ar : 0.0, on ? v.ai : 0.0, on ? v.br : 0.0, on ? v.bi : 0.0};
}

__device__ __forceinline__ double flip_sign(double v, unsigned mask) {
  return mkd(lo32(v), hi32(v) ^ mask);
}

template <class T, bool ACT, bool BCT>
__device__ __forceinline__ void qgemm2_tile(const QGemmTask& t, int row0, int col0, int kbeg, int kend, quat* C) {
  constexpr int TBM = T::TBM, TBN = T::TBN, GBK = T::GBK;
  constexpr int AH = TBM * GBK / 256;   // A stage elements per thread
  constexpr int BH = TBN * GBK / 256;   // B stage elements per thread
  constexpr int WM = T::WM, WN = 4 / WM;
  constexpr int WR = TBM / WM, WC = TBN / WN;   // quaternion rows and columns per wave
  constexpr int NA = WR / 4, NBC = WC / 16;   // MFMA accumulators per wave: NA x NBC
  static_assert(AH * 256 == TBM * GBK && BH * 256 == TBN * GBK && NA * 4 == WR && NBC * 16 == WC, "tile shape");
  const int m = t.m, nn = t.nn;
  __shared__ double As[2][GBK * T::ASK];
  __shared__ double Bs[2][GBK * T::BSK];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  const int wr = wv / WN, wc = wv % WN;   // wave tile: rows wr*WR..+WR, cols wc*WC..+WC (quaternions)
  const int cr = (lane & 15) >> 2, ck = lane >> 4;
  const int acomp = cr ^ ck;
  const unsigned smask = ((0x428E >> (cr * 4 + ck)) & 1) ? 0x80000000u : 0u;
  const int aq = lane & 3;
  const int bkc = lane >> 4, bj = lane & 15;
  // this thread's A and B stage elements: consecutive threads along the
  // storage's contiguous direction
  int ai[AH], ak[AH], bk[BH], bjj[BH];
#pragma unroll
  for (int h = 0; h < AH; ++h) {
    if (!ACT) { ai[h] = tid % TBM; ak[h] = tid / TBM + (256 / TBM) * h; }
    else { ak[h] = tid % GBK; ai[h] = tid / GBK + (256 / GBK) * h; }
  }
#pragma unroll
  for (int h = 0; h < BH; ++h) {
    if (!BCT) { bk[h] = tid % GBK; bjj[h] = tid / GBK + (256 / GBK) * h; }
    else { bjj[h] = tid % TBN; bk[h] = tid / TBN + (256 / TBN) * h; }
  }
  quat ra[AH], rb[BH];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int h = 0; h < AH; ++h) ra[h] = ld_op<ACT>(t.A, min(row0 + ai[h], m - 1), min(k0 + ak[h], kend - 1));
#pragma unroll
    for (int h = 0; h < BH; ++h) rb[h] = ld_op<!BCT>(t.B, min(col0 + bjj[h], nn - 1), min(k0 + bk[h], kend - 1));
  };
  auto stash = [&](int buf, int k0) {
#pragma unroll
    for (int h = 0; h < AH; ++h) {
      const int i = row0 + ai[h], k = k0 + ak[h];
      const quat a = qselect(i < m && k < kend && op_on<ACT>(t.A, i, k), ACT ? qconj(ra[h]) : ra[h]);
      double2* pa = reinterpret_cast<double2*>(&As[buf][ak[h] * T::ASK + ai[h] * 4]);
      pa[0] = make_double2(a.ar, a.ai);
      pa[1] = make_double2(a.br, a.bi);
    }
#pragma unroll
    for (int h = 0; h < BH; ++h) {
      const int j = col0 + bjj[h], k = k0 + bk[h];
      const quat bv = qselect(j < nn && k < kend && op_on<!BCT>(t.B, j, k), BCT ? qconj(rb[h]) : rb[h]);
      double* pb = &Bs[buf][bk[h] * T::BSK + bjj[h]];
      pb[0] = bv.ar;
      pb[TBN] = bv.ai;
      pb[2 * TBN] = bv.br;
      pb[3 * TBN] = bv.bi;
    }
  };
  // lane holds quaternion (row wr*WR + 4a + lane/16, col wc*WC + 16b + lane%16) of C
  const double alpha = t.alpha, beta = t.beta;
  const int ci = row0 + wr * WR + (lane >> 4), cj = col0 + wc * WC + (lane & 15);
  auto written = [&](int a, int b) {
    const int i = ci + 4 * a, jj = cj + 16 * b;
    return i < m && jj < nn && (!t.lower_only || i >= jj);
  };
  quat cold[T::PREC ? NA : 1][T::PREC ? NBC : 1];
  if constexpr (T::PREC) {
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int b = 0; b < NBC; ++b) {
        cold[a][b] = qzero();
        if (beta != 0.0 && written(a, b)) cold[a][b] = qload_g(C + (ci + 4 * a) + (size_t)(cj + 16 * b) * t.ldc);
      }
  }
  d4 acc[NA][NBC];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NBC; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
  int cur = 0;
  if (kbeg < kend) {
    fetch(kbeg);
    stash(0, kbeg);
  }
  __syncthreads();
  for (int k0 = kbeg; k0 < kend; k0 += GBK) {
    const bool more = k0 + GBK < kend;
    if (more) fetch(k0 + GBK);
#pragma unroll
    for (int kk = 0; kk < GBK; ++kk) {
      double af[NA], bf[NBC];
#pragma unroll
      for (int a = 0; a < NA; ++a) af[a] = flip_sign(As[cur][kk * T::ASK + (wr * WR + 4 * a + aq) * 4 + acomp], smask);
#pragma unroll
      for (int b = 0; b < NBC; ++b) bf[b] = Bs[cur][kk * T::BSK + bkc * TBN + wc * WC + 16 * b + bj];
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < NBC; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
    if (more) stash(cur ^ 1, k0 + GBK);
    __syncthreads();
    cur ^= 1;
  }
#pragma unroll
  for (int a = 0; a < NA; ++a) {
#pragma unroll
    for (int b = 0; b < NBC; ++b) {
      if (written(a, b)) {
        quat* cp = C + (ci + 4 * a) + (size_t)(cj + 16 * b) * t.ldc;
        quat r = quat{alpha * acc[a][b][0], alpha * acc[a][b][1], alpha * acc[a][b][2], alpha * acc[a][b][3]};
        if (beta != 0.0) r = qaxpy(r, beta, T::PREC ? cold[T::PREC ? a : 0][T::PREC ? b : 0] : qload_g(cp));
        qstore_g(cp, r);
      }
    }
  }
}

// Workgroups are dealt to the 8 XCDs round-robin by launch order.  The tile
// index is remapped so that each XCD works through a contiguous range of
// tiles (column-major over the tile grid), which share operand tiles in its
// L2: XCD k = t mod 8 owns floor(T/8) (+1 for k < T mod 8) consecutive ones.
__device__ __forceinline__ int xcd_remap(int t, int T) {
  const int k = t & 7;
  return k * (T >> 3) + min(k, T & 7) + (t >> 3);
}

// Lower-triangle products enumerate only the tiles that meet the lower
// triangle: column block y (TBN wide) has row tiles x >= y TBN / TBM, so the
// blocks before it hold y gx - (TBN / TBM) y (y - 1) / 2 tiles.
template <class T>
__host__ __device__ inline int tiles_before(int y, int gx) {
  static_assert(T::TBN % T::TBM == 0, "lower-triangle tile enumeration");
  return y * gx - T::TBN / T::TBM * (y * (y - 1) / 2);
}
template <class T>
__host__ __device__ inline int tile_count(int m, int nn, bool lower) {
  const int gx = (m + T::TBM - 1) / T::TBM, gy = (nn + T::TBN - 1) / T::TBN;
  return lower ? tiles_before<T>((m + T::TBN - 1) / T::TBN, gx) : gx * gy;
}

template <class T>
__device__ __forceinline__ void tile_of(const QGemmTask& t, int u, int& tx, int& ty) {
  const int gx = (t.m + T::TBM - 1) / T::TBM;
  if (!t.lower_only) {
    ty = u / gx;
    tx = u - ty * gx;
    return;
  }
  // the largest y with tiles_before(y) <= u: the root of the quadratic, then exact
  constexpr int rho = T::TBN / T::TBM;
  const float bq = 2.0f * (float)gx / rho + 1.0f;
  int y = (int)(0.5f * (bq - sqrtf(fmaxf(bq * bq - 8.0f / rho * (float)u, 0.0f))));
  const int gy = (t.m + T::TBN - 1) / T::TBN;
  y = max(0, min(y, gy - 1));
  while (y + 1 < gy && tiles_before<T>(y + 1, gx) <= u) ++y;
  while (y > 0 && tiles_before<T>(y, gx) > u) --y;
  ty = y;
  tx = rho * y + (u - tiles_before<T>(y, gx));
}

// grid: x = tiles, z = K chunks
template <class T, bool ACT, bool BCT>
__global__ void __launch_bounds__(256, 2) k_qgemm2(QGemmTask t, int kchunk, size_t cstride) {
  int tx, ty;
  tile_of<T>(t, xcd_remap(blockIdx.x, gridDim.x), tx, ty);
  int kbeg = t.kbeg, kend = t.kend;
  quat* C = t.C;
  if (gridDim.z > 1) {
    kbeg = t.kbeg + blockIdx.z * kchunk;
    kend = min(t.kend, kbeg + kchunk);
    C += (size_t)blockIdx.z * cstride;
  }
  qgemm2_tile<T, ACT, BCT>(t, tx * T::TBM, ty * T::TBN, kbeg, kend, C);
}

// grid: x = tiles of the largest task, z = tasks; with nfold tasks folded, x =
// tiles of the largest pair, and row z holds the tiles of tasks z and nfold - 1 - z
template <class T, bool ACT, bool BCT>
__global__ void __launch_bounds__(256, 2) k_qgemm2_batch(const QGemmTask* __restrict__ tasks, int nfold) {
  int z = blockIdx.z;
  int u = xcd_remap(blockIdx.x, gridDim.x);
  const int z2 = nfold > 0 ? nfold - 1 - z : z;
  const int nt = tile_count<T>(tasks[z].m, tasks[z].nn, tasks[z].lower_only);
  const int nt2 = tile_count<T>(tasks[z2].m, tasks[z2].nn, tasks[z2].lower_only);
  if (u >= nt) {
    u -= nt;
    if (z2 == z || u >= nt2) return;
    z = z2;
  }
  const QGemmTask t = tasks[z];
  int tx, ty;
  tile_of<T>(t, u, tx, ty);
  qgemm2_tile<T, ACT, BCT>(t, tx * T::TBM, ty * T::TBN, t.kbeg, t.kend, t.C);
}

// Tile rows: 64 only for launches with at least 16 64 x 64 tiles per compute
// unit, else 32 (twice the workgroups: better balance and register use).
// Measured on the 2n = 8192 solve, each step against the previous one on
// one box: switch at 2 -> 4 tiles per CU -0.6 ms, 4 -> 8 -1.5 ms, 8 -> 16
// -0.9 ms; 32 rows always is equal to 16 within noise; the batch of 512
// problems stays within 0.5%.
static int device_cus() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (!cached[dev]) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    cached[dev] = cus;
  }
  return cached[dev];
}

thread_local int g_tile64_per_cu = 16;

// 16 x 32 tiles for launches of fewer than SMALL_PER_CU 32 x 64 tiles per
// compute unit.  Against 32 x 64 tiles throughout (2n = 510, 1024, 2048, 4096
// solves 2.55, 5.13, 11.25, 33.8 ms): below 1 tile per unit 2.31, 4.66, 10.83,
// 33.4 ms, below 2 2.30, 4.65, 10.78, 33.2 ms, below 4 2.30, 4.65, 10.82, 33.8
// ms, below 8 the 2n = 8192 solve too is slower (149.0 -> 151.9 ms): more
// operand traffic per product once every CU is busy.
// And of at most SMALL_ROUNDS 16 x 32 tiles per unit: a launch's time goes by the
// tiles of its fullest unit, and 8 small ones take longer than the 2 large ones
// that a full round holds.  16 x 32 over 32 x 64, K = 16, 64, 256, 1024: at 5
// tiles per unit 0.71, 0.72, 0.70, 0.70, at 6 0.80, 0.82, 0.83, 0.83, at 7 0.87,
// 0.93, 0.96, 0.97, at 8 0.92, 1.03, 1.09, 1.10 (960 x 1000 x 1000: 541 and 598 us).
constexpr int SMALL_PER_CU = 2, SMALL_ROUNDS = 7;
static int tile_rows(long tiles64, long tiles32, long tiles16) {
  if (tiles32 < (long)SMALL_PER_CU * device_cus() && tiles16 <= (long)SMALL_ROUNDS * device_cus()) return 16;
  return tiles64 >= (long)g_tile64_per_cu * device_cus() ? 64 : 32;
}

template <class T>
static void launch_gemm2_t(bool act, bool bct, hipStream_t s, const QGemmTask& t, int nz, int kchunk,
                           size_t cstride) {
  const dim3 grid(tile_count<T>(t.m, t.nn, t.lower_only), 1, nz);
  if (!act && !bct) launch_k(k_qgemm2<T, false, false>, grid, dim3(256), 0, s, t, kchunk, cstride);
  else if (act && !bct) launch_k(k_qgemm2<T, true, false>, grid, dim3(256), 0, s, t, kchunk, cstride);
  else if (!act && bct) launch_k(k_qgemm2<T, false, true>, grid, dim3(256), 0, s, t, kchunk, cstride);
  else launch_k(k_qgemm2<T, true, true>, grid, dim3(256), 0, s, t, kchunk, cstride);
}

static void launch_gemm2(bool act, bool bct, hipStream_t s, const QGemmTask& t, int nz, int kchunk, size_t cstride) {
  const bool low = t.lower_only;
  switch (tile_rows((long)tile_count<Tile64>(t.m, t.nn, low) * nz, (long)tile_count<Tile32>(t.m, t.nn, low) * nz,
                    (long)tile_count<Tile16>(t.m, t.nn, low) * nz)) {
    case 64: launch_gemm2_t<Tile64>(act, bct, s, t, nz, kchunk, cstride); break;
    case 32:
      if (low) launch_gemm2_t<Tile32L>(act, bct, s, t, nz, kchunk, cstride);
      else launch_gemm2_t<Tile32>(act, bct, s, t, nz, kchunk, cstride);
      break;
    default: launch_gemm2_t<Tile16>(act, bct, s, t, nz, kchunk, cstride); break;
  }
}

// A list's tasks differ in size (a batch's members, largest first): with one row
// of blocks per task, as long as the largest task's, more than half of a
// batch's blocks were empty, and each holds an LDS allocation until it has read
// its task.  Tasks z and ntasks - 1 - z share a row where that takes fewer
// blocks (batch of 512 72.7 -> 72.3 ms, 2n = 8192 solve 145.4 -> 145.2 ms).
// tasks_host: the same list.
template <class T>
static void launch_gemm2_batch_t(bool act, bool bct, int ntasks, int tiles, hipStream_t s, const QGemmTask* tasks,
                                 const QGemmTask* tasks_host) {
  const int w = fold_width(ntasks, [&](int z) {
    return tile_count<T>(tasks_host[z].m, tasks_host[z].nn, tasks_host[z].lower_only);
  });
  const int rows = (ntasks + 1) / 2;
  const bool fold = (long)w * rows < (long)tiles * ntasks;
  const int nfold = fold ? ntasks : 0;
  const dim3 grid(fold ? w : tiles, 1, fold ? rows : ntasks);
  if (!act && !bct) launch_k(k_qgemm2_batch<T, false, false>, grid, dim3(256), 0, s, tasks, nfold);
  else if (act && !bct) launch_k(k_qgemm2_batch<T, true, false>, grid, dim3(256), 0, s, tasks, nfold);
  else if (!act && bct) launch_k(k_qgemm2_batch<T, false, true>, grid, dim3(256), 0, s, tasks, nfold);
  else launch_k(k_qgemm2_batch<T, true, true>, grid, dim3(256), 0, s, tasks, nfold);
}

int qgemm(int m, int nn, int k, double alpha, const QOperand& A, const QOperand& B, double beta, quat* C, int ldc,
          bool lower_only, hipStream_t s) {
  if (m <= 0 || nn <= 0) return ZQI_OK;
  QGemmTask t{m, nn, 0, k, ldc, lower_only ? 1 : 0, alpha, beta, A, B, C};
  launch_gemm2(A.conj_trans, B.conj_trans, s, t, 1, k, (size_t)0);
  return hipGetLastError() == hipSuccess ? ZQI_OK : ZQI_ERR_HIP;
}

// Task lists of split-K chunks of at least LONG_K (but for a sum's last chunk)
// take 64-row tiles already from two per CU, where they all run at once: the
// back-transform's Y products at n >= 4096 (1024 32-row tiles make one and a third
// rounds of three per CU, 512 64-row ones one round of two; 2n = 8192
// back-transform 39.3 -> 38.4 ms).
constexpr int LONG_K = 384;
int qgemm_tasks(const QGemmTask* tasks_dev, const QGemmTask* tasks_host, int ntasks, int maxm, int maxnn, int kchunk,
                bool act, bool bct, bool lower, hipStream_t s) {
  if (ntasks <= 0 || maxm <= 0 || maxnn <= 0) return ZQI_OK;
  const int n64 = tile_count<Tile64>(maxm, maxnn, lower), n32 = tile_count<Tile32>(maxm, maxnn, lower);
  // 64-row tiles by the largest task alone: many smaller ragged tasks lose more
  // to the padding of their edges than the larger tiles save (the 512-problem
  // batch 70.3 ms counting all tasks' tiles, 68.8 ms so)
  int rows = tile_rows((long)n64, (long)n32 * ntasks, (long)tile_count<Tile16>(maxm, maxnn, lower) * ntasks);
  if (rows == 32 && kchunk >= LONG_K && (long)n64 * ntasks >= 2L * device_cus()) rows = 64;
  switch (rows) {
    case 64: launch_gemm2_batch_t<Tile64>(act, bct, ntasks, n64, s, tasks_dev, tasks_host); break;
    case 32:
      if (lower)
        launch_gemm2_batch_t<Tile32L>(act, bct, ntasks, tile_count<Tile32L>(maxm, maxnn, lower), s, tasks_dev,
                                      tasks_host);
      else
        launch_gemm2_batch_t<Tile32>(act, bct, ntasks, n32, s, tasks_dev, tasks_host);
      break;
    default:
      launch_gemm2_batch_t<Tile16>(act, bct, ntasks, tile_count<Tile16>(maxm, maxnn, lower), s, tasks_dev, tasks_host);
  }
  return hipGetLastError() == hipSuccess ? ZQI_OK : ZQI_ERR_HIP;
}

// Split-K chunks: multiples of KCHUNK, and not shorter than KCHUNK_MIN: below
// that the partials' traffic and the launch that sums them cost more than the
// split saves (batch of 512 problems 74.7 ms with chunks from 16, 74.1 from 64,
// 73.5 from 128; 2n = 510 solve 2.03, 2.03, 2.05 ms).
constexpr int KCHUNK = 16, KCHUNK_MIN = 64;
int splitk_count(int K, int nsplit, int* kchunk_out) {
  if (nsplit < 1) nsplit = 1;
  int kchunk = (K + nsplit - 1) / nsplit;
  kchunk = std::max(((kchunk + KCHUNK - 1) / KCHUNK) * KCHUNK, KCHUNK_MIN);
  if (kchunk_out) *kchunk_out = kchunk;
  const int nz = (K + kchunk - 1) / kchunk;
  return nz > 0 ? nz : 1;
}

// ---------------------------------------------------------------------------
// Real FP64 GEMM for the divide & conquer merges of one tree level, one merge
// per blockIdx.z: for the merge of rows [lo, hi) (ns = hi - lo) of problem
// base ob,  Z[lo:hi, lo - ob + posK[j]] = Qtmp_m (ns x K) U_m (K x K), with
// K = kcnt[z] read on the device (data-dependent after deflation) and the
// merge's Qtmp / U blocks at lo * lq (ld ns).  Qtmp's columns come in three
// groups: [0, g0) hold rows of the first half (rows < mid - lo) only, [g0,
// g1) both halves, [g1, K) the second half only (kgrp[2z], kgrp[2z + 1]), so
// a tile of first-half rows sums over [0, g1) and one of second-half rows
// over [g0, K), skipping exact zeros (as LAPACK's dlaed3 splits the product).
// ---------------------------------------------------------------------------
constexpr int DBM = 64, DBN = 64, DBK = 16;

// 64 x 64 tile per workgroup (2 x 2 waves of 32 x 32), K staged 16 at a time
// through double-buffered LDS; the next stage's operands are fetched into
// registers before the current stage's MFMAs (one barrier per stage).
__global__ void __launch_bounds__(256) k_dgemm_merge(const MergeDesc* __restrict__ descs, const int* __restrict__ kcnt,
                                                     const int* __restrict__ kgrp, const double* __restrict__ Qtmp,
                                                     const double* __restrict__ U, int lq, double* __restrict__ Z,
                                                     int ldz, const int* __restrict__ posK,
                                                     const int* __restrict__ posD) {
  const MergeDesc md = descs[blockIdx.z];
  const int K = kcnt[blockIdx.z];
  const int m = md.hi - md.lo, n1 = md.mid - md.lo;
  const int row0 = blockIdx.x * DBM, col0 = blockIdx.y * DBN;
  if (col0 >= m || row0 >= m) return;
  if (col0 + DBN > K) {
    // columns K .. of Qtmp are the deflated ones: copied to their final columns
    const int i = row0 + (threadIdx.x & (DBM - 1));
    if (i < m)
      for (int j = max(col0, K) + (threadIdx.x >> 6); j < min(col0 + DBN, m); j += 4)
        Z[md.lo + i + (size_t)(md.lo - md.ob + posD[md.lo + j - K]) * ldz] =
            Qtmp[(size_t)md.lo * lq + i + (size_t)j * m];
    if (col0 >= K) return;
  }
  // the sum's range for this tile's rows (the full range for a tile across the halves)
  const int kb = row0 >= n1 ? kgrp[2 * blockIdx.z] : 0;
  const int ke = row0 + DBM <= n1 ? kgrp[2 * blockIdx.z + 1] : K;
  const double* A = Qtmp + (size_t)md.lo * lq;
  const double* B = U + (size_t)md.lo * lq;
  const int lda = m, ldb = m;
  double* C = Z + md.lo + (size_t)(md.lo - md.ob) * ldz;
  const int* cmap = posK + md.lo;
  __shared__ double As[2][DBK][DBM + 1];
  __shared__ double Bs[2][DBK][DBN + 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wr = wv >> 1, wc = wv & 1;  // 32 x 32 per wave
  constexpr int NE = DBK * DBM / 256;   // stage elements per thread and operand
  double ra[NE], rb[NE];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int h = 0; h < NE; ++h) {
      const int idx = tid + 256 * h;
      const int i = idx & (DBM - 1), k = idx >> 6;
      const int gi = row0 + i, gk = k0 + k;
      ra[h] = (gi < m && gk < ke) ? A[gi + (size_t)gk * lda] : 0.0;
      const int kr = idx & (DBK - 1), jb = idx / DBK;
      const int gkb = k0 + kr, gj = col0 + jb;
      rb[h] = (gkb < ke && gj < K) ? B[gkb + (size_t)gj * ldb] : 0.0;
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int h = 0; h < NE; ++h) {
      const int idx = tid + 256 * h;
      As[buf][idx >> 6][idx & (DBM - 1)] = ra[h];
      Bs[buf][idx & (DBK - 1)][idx / DBK] = rb[h];
    }
  };
  d4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
  fetch(kb);
  stash(0);
  __syncthreads();
  int cur = 0;
  for (int k0 = kb; k0 < ke; k0 += DBK) {
    const bool more = k0 + DBK < ke;
    if (more) fetch(k0 + DBK);
#pragma unroll
    for (int kk = 0; kk < DBK; kk += 4) {
      double af[2], bf[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) af[a] = As[cur][kk + (lane >> 4)][wr * 32 + 16 * a + (lane & 15)];
#pragma unroll
      for (int b = 0; b < 2; ++b) bf[b] = Bs[cur][kk + (lane >> 4)][wc * 32 + 16 * b + (lane & 15)];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
    if (more) stash(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int j = col0 + wc * 32 + 16 * b + (lane & 15);
      if (j >= K) continue;
      const int cj = cmap[j];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = row0 + wr * 32 + 16 * a + 4 * r + (lane >> 4);
        if (i < m) C[i + (size_t)cj * ldz] = acc[a][b][r];
      }
    }
}

int dgemm_merges(const MergeDesc* descs_dev, int nmerge, int nsmax, const int* kcnt, const int* kgrp,
                 const double* Qtmp, const double* U, int lq, double* Z, int ldz, const int* posK, const int* posD,
                 hipStream_t s) {
  if (nmerge <= 0 || nsmax <= 0) return ZQI_OK;
  dim3 grid((nsmax + DBM - 1) / DBM, (nsmax + DBN - 1) / DBN, nmerge);
  launch_k(k_dgemm_merge, grid, dim3(256), 0, s, descs_dev, kcnt, kgrp, Qtmp, U, lq, Z, ldz, posK, posD);
  return hipGetLastError() == hipSuccess ? ZQI_OK : ZQI_ERR_HIP;
}

// Raw MFMA probe: D = A (16x4) B (4x16) with lane-indexed inputs; used by the
// self-test that pins the register layout the kernels above assume.
__global__ void k_mfma_probe(const double* a, const double* b, double* out) {
  const int l = threadIdx.x;
  d4 acc = d4{0.0, 0.0, 0.0, 0.0};
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[l], b[l], acc, 0, 0, 0);
  for (int r = 0; r < 4; ++r) out[l * 4 + r] = acc[r];
}

int mfma_probe(const double* a, const double* b, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, s, a, b, out);
  return hipGetLastError() == hipSuccess ? ZQI_OK : ZQI_ERR_HIP;
}

}  // namespace zq
