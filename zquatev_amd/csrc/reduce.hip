// Quaternion Householder tridiagonalisation (the panel and trailing update).
//
// Replaces the reference's symplectic reduction: impl::panel_update
// (blocked.cc:45-546) and impl::unblocked_update (unblocked.cc:44-131), driven
// by the panel loop at zquatev.cc:68-72.  The reference applies three complex
// symplectic transforms per column (a B-column Householder, a Givens rotation
// between the A and B blocks, an A-column Householder).  Here one quaternion
// Householder reflector H = I - u u^* (u^* u = 2) clears column c of the
// quaternion matrix M below its subdiagonal in one step; by the implicit-Q
// theorem the real tridiagonal obtained after the diagonal phase scaling is
// the same one the reference hands to zhbev (zquatev.cc:74-84).
//
// Blocked (latrd-style) form: within a panel of nb columns starting at p the
// trailing matrix is M - V W^* - W V^*, where V holds the panel's reflectors
// (stored in place below the subdiagonal of M) and
//   w_j = p_j - (u_j^* p_j / 2) u_j,   p_j = M u_j - V (W^* u_j) - W (V^* u_j).
// After the panel, the trailing lower triangle gets the rank-2nb update on
// FP64 MFMA (gemm.hip).  Per column the only pass over the trailing matrix is
// the Hermitian matvec M u_j, which reads the lower triangle once (16 m^2
// bytes for an m x m trailing block).
#include "zq_internal.h"
#include <climits>
#include <algorithm>
#include <vector>

namespace zq {

constexpr int RB = 256;      // threads per block of the row kernels
constexpr int RQ = 16;       // rows per block of the row kernels (16 threads per row split the K sums)
constexpr int SG = 64;       // matvec rows per block (one per lane)
// Matvec tile shapes: SG rows x SW columns.  Trailing sizes up to the switch
// tsm use narrow strips (SW = 16, 256 threads: more, smaller blocks, which
// keeps the small matvecs of batches and of the end of a solve spread over
// the CUs); larger ones wide strips (SW = 32, 512 threads: fewer row
// partials for the column kernel to gather).  spg = SG / SW strips per row
// group.  The switch is a per-context tuning parameter (0 .. TSM_MAX; the
// autotuner times candidates), 768 by default.
constexpr int TSM_MAX = 2048;
__host__ __device__ constexpr int matvec_spg(int m, int tsm) { return m <= tsm ? 4 : 2; }
// matvec tiles of a trailing size with G row groups: group g holds spg (g + 1) strips
__host__ __device__ constexpr int ntiles(int G, int spg) { return spg * G * (G + 1) / 2; }
// blocks of k_symv (nf of them finishing blocks) and of k_wcol at trailing size sz
__host__ __device__ constexpr int symv_blocks(int sz, int spg, int nf) { return ntiles((sz + SG - 1) / SG, spg) + nf; }
__host__ __device__ constexpr int wcol_blocks(int sz) { return sz - 1 > RQ ? (sz - 1 + RQ - 1) / RQ : 1; }
constexpr int NBMAX = 128;   // largest supported panel width
constexpr int TAILN = 64;    // trailing size from which one workgroup finishes (k_tail)

// ceil(a / b) for b > 0, and 0 for a <= 0
__device__ __forceinline__ int cdiv_d(int a, int b) { return a > 0 ? (a + b - 1) / b : 0; }

__device__ __forceinline__ double block_sum(double v, double* sh) {
  v = wave_sum_d(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  const int nw = (blockDim.x + 63) >> 6;
  for (int i = 0; i < nw; ++i) r += sh[i];
  __syncthreads();
  return r;
}

// Whether an entry of the tridiagonal's first c columns exceeds v (one thread)
__device__ __forceinline__ bool any_above(const double* d, const quat* e, int c, double v) {
  for (int k = 0; k < c; ++k)
    if (fabs(d[k]) > v || qabs(qload(e + k)) > v) return true;
  return false;
}

// Reflector for column c: x = M[c+1:, c].  H x = alpha e_1 with
// alpha = -q |x|, q = x_1/|x_1|; u = gamma (x - alpha e_1), gamma = 1/sqrt(|x| (|x| + |x_1|)),
// so u^* u = 2.  A zero tail gives u = 0 and alpha = x_1.  Computed identically
// by every block that needs it.
struct Refl {
  double g;
  quat u1;
};
__device__ __forceinline__ Refl reflector(const quat& x1, double tail, quat* alpha) {
#pragma clang fp contract(off)
  // the two square roots and the reciprocal do not wait for each other
  const double x2 = qnorm2(x1);
  const double ax1 = sqrt(x2), nx = sqrt(x2 + tail), ix1 = rsqrt(x2);
  Refl R;
  if (!(tail > 0.0)) {
    R.g = 0.0;
    R.u1 = qzero();
    *alpha = x1;
  } else {
    const quat qph = (ax1 > 0.0) ? qscale(x1, ix1) : quat{1.0, 0.0, 0.0, 0.0};
    const double sm = ax1 + nx;
    R.g = rsqrt(nx * sm);
    R.u1 = qscale(qph, sm * R.g);
    *alpha = qscale(qph, -nx);
  }
  return R;
}


// Hermitian matvec over the lower triangle of the trailing matrix
// M[s0:, s0:] (s0 = c + 1), applied to the raw updated column x = M[s0:, c]
// rather than to the reflector u: u = gamma x + (u1 - gamma x1) e_1, so
//   M u = gamma (M x) + (u1 - gamma x1) M[s0:, s0],
// which k_wcol forms row by row.  The tile blocks therefore never wait for
// the reflector (no norm reduction on their path).  Each tile block also
// leaves its share of x^* M x (the lower part doubled off the diagonal) in
// QF[b], from which k_wcol forms u^* M u without another grid-wide reduction.
// Block (g, J) reads rows [s0 + SG g, +SG) x columns [s0 + SW J, +SW) (every
// lower-triangle element exactly once over the grid); wave w of NWV takes SCW of
// the SW columns, one row per lane, all loads issued up front.  Row sums over
// the SW columns (summed across the waves in LDS) go to Prow[J][row]; column
// sums over the SG rows (a VALU-only halving butterfly, DPP and permlane
// swaps) go to Pcol[g][col]; then
//   (M x)(i) = sum_{J <= (i-s0)/SW} Prow[J][i] + sum_{g >= (i-s0)/SG} Pcol[g][i],
// every (slot, row) written exactly once, so the sum is deterministic.
// Blocks are enumerated row-group major: group g has SPG (g + 1) strips.
// The max(1, ceil(8 j / 64)) blocks before the ntiles(G) tiles compute the
// reflector from the tail-norm partials (from the column itself for a
// panel's first column, j = 0) (the first of them publishes gamma,
// u1, x1 in scal and d[c], e[c]) and finish the tall-skinny products
// TS = [W^* u | V^* u]: they add the per-block partials of W^* x and V^* x
// that k_wcol left in TSP (the waves over the partial index, then the
// wave sums, in a fixed order), scale by gamma and add the row s0 term.
template <int SYT, int SW, bool BT>
__global__ void __launch_bounds__(SYT) k_symv(
    const quat* __restrict__ M, const quat* __restrict__ W, const double* __restrict__ TSP,
    const double* __restrict__ part, int ld, int n, int p, int c, int j, int ldw, int nparts, int ldtsp,
    double* __restrict__ scal, double* __restrict__ d, quat* __restrict__ e, quat* __restrict__ Prow,
    quat* __restrict__ Pcol, int ldp, int nb, quat* __restrict__ TS, double* __restrict__ QF, ZB zb) {
  constexpr int NWV = SYT / 64;    // waves per block
  constexpr int SCW = SW / NWV;     // strip columns per wave
  constexpr int SPG = SG / SW;      // strips per row group and group index
  static_assert(SW <= SG && SG % SW == 0 && SW % NWV == 0, "matvec tile shape");
  const int NT = j > 0 ? (8 * j + 63) / 64 : 0;
  const int NF = NT > 0 ? NT : 1;
  int bt = blockIdx.x;
  if constexpr (BT) {
    int z;
    if (!fold_member(zb, [=](int m) { return symv_blocks(m - c - 1, SPG, NF); }, z, n, bt)) return;
    nparts = (n - c - 1 + RQ - 1) / RQ;
    M = zoff(M, zb, z); W = zoff(W, zb, z); part = zoff(part, zb, z); scal = zoff(scal, zb, z); d = zoff(d, zb, z);
    e = zoff(e, zb, z); Prow = zoff(Prow, zb, z); Pcol = zoff(Pcol, zb, z); TS = zoff(TS, zb, z);
    TSP = zoff(TSP, zb, z); QF = zoff(QF, zb, z);
  }
  __shared__ double sh[SYT / 64];
  __shared__ double sqf[SYT / 64];
  __shared__ double red[NWV][4][SG];   // wave, component, row: conflict-free b64 accesses
  const int s0 = c + 1;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: its column loads are scalar
  // blocks [0, NF) finish the column (dispatched first, so they overlap the
  // tiles), blocks NF + b take tile b
  const int b = bt - NF;
  if (b < 0) {
    // ---- finishing block: reflector, scalars, tall-skinny products
    const bool has_ts = bt < NT;
    // the row-s0 entries of W and V (for the u_1 term of TS), the diagonal
    // entries, and the partials in batches of 8 per lane
    const int e0 = 64 * bt + 4 * (tid & 15);
    const int lts = e0 >> 3, side = (e0 >> 2) & 1;
    const bool fin = has_ts && tid < 16 && lts < j;
    quat rowv = qzero();
    if (fin) rowv = side == 0 ? qload(W + s0 + (size_t)lts * ldw) : qload(M + s0 + (size_t)(p + lts) * ld);
    double mss = 0.0, mcc = 0.0;
    if (bt == 0 && tid == 0) {
      mss = M[s0 + (size_t)s0 * ld].ar;
      if (j == 0) mcc = M[c + (size_t)c * ld].ar;
    }
    const quat x1 = qload(M + s0 + (size_t)c * ld);
    double tail = 0.0, tsacc = 0.0;
    if (has_ts) {
      // the tail norm from the partials the column kernel left, in wave 0 alone
      // (it and its reflector then wait for no other wave)
      if (w == 0)
        for (int k = lane; k < nparts; k += 64) tail += part[k];
      const int eidx = 64 * bt + lane;
      constexpr int TB = 8;
      for (int k0 = w; k0 < nparts; k0 += NWV * TB) {
        double v[TB];
#pragma unroll
        for (int u = 0; u < TB; ++u) v[u] = TSP[(size_t)min(k0 + NWV * u, nparts - 1) * ldtsp + eidx];
#pragma unroll
        for (int u = 0; u < TB; ++u) tsacc = fma(k0 + NWV * u < nparts ? 1.0 : 0.0, v[u], tsacc);
      }
      tail = wave_sum_d(tail);
    } else {   // a panel's first column has no pending update: its tail norm from the column itself
      for (int i = c + 2 + tid; i < n; i += SYT) tail += qnorm2(qload(M + i + (size_t)c * ld));
      tail = block_sum(tail, sh);
    }
    // A column whose squares lose digits counts as reduced (u = 0): it is at most
    // 1e-140, and neither its norm nor x^* M x is known.  One that is not zero and
    // below the reach of gamma^2 is told apart from a matrix of that scale, which
    // this reduction cannot take (not finite, as its gamma^2), by a larger entry of
    // d or e so far.
    const double s = qnorm2(x1) + tail;
    const bool drop = s < TINY_SQ;
    quat alpha;
    const Refl R = reflector(x1, drop ? 0.0 : tail, &alpha);
    if (bt == 0 && tid == 0) {
      if (drop && s > 0.0 && s < 3e-309 && !any_above(d, e, c, 1e-130)) alpha.ar = __builtin_nan("");
      scal[0] = R.g;
      scal[1] = R.u1.ar; scal[2] = R.u1.ai; scal[3] = R.u1.br; scal[4] = R.u1.bi;
      scal[5] = x1.ar; scal[6] = x1.ai; scal[7] = x1.br; scal[8] = x1.bi;
      scal[9] = mss;   // M[s0, s0]
      if (j == 0) d[c] = mcc;   // inside a panel the column kernel has left d[c]
      qstore(e + c, alpha);
    }
    if (has_ts) {
      __shared__ double tsr[NWV][64];
      tsr[w][lane] = tsacc;
      __syncthreads();
      // quaternion (side, l) = entries 64 bt + 4 tid .. + 3, entry index 8 l + 4 side + component
      if (fin) {
        double sc[4];
#pragma unroll
        for (int comp = 0; comp < 4; ++comp) {
          double t = 0.0;
#pragma unroll
          for (int k = 0; k < NWV; ++k) t += tsr[k][4 * tid + comp];
          sc[comp] = t;
        }
        quat t = qscale(quat{sc[0], sc[1], sc[2], sc[3]}, R.g);
        qfma_cl(t, rowv, R.u1);
        qstore(TS + (size_t)side * nb + lts, t);
      }
    }
    return;
  }
  // ---- tile block: block -> (g, J) with ntiles(g) <= b < ntiles(g + 1)
  int g = (int)((sqrtf(8.0f / SPG * (float)b + 1.0f) - 1.0f) * 0.5f);   // corrected below
  while (ntiles(g + 1, SPG) <= b) ++g;
  while (ntiles(g, SPG) > b) --g;
  const int J = b - ntiles(g, SPG);
  const int R0 = s0 + SG * g, C0 = s0 + SW * J;
  const bool active = C0 < n && R0 < n;   // uniform for the block
  const int ra = R0 + lane;
  const int rac = min(ra, n - 1);
  // Above the diagonal (row < column: unused, masked below) a lane reads the
  // column's diagonal entry instead, a line the tile fetches anyway, so the
  // diagonal tiles' upper halves cost no memory traffic and no branch.
  quat qa[SCW];
#pragma unroll
  for (int cc = 0; cc < SCW; ++cc) {
    const int cgc = min(C0 + SCW * w + cc, n - 1);
    qa[cc] = qload(M + max(rac, cgc) + (size_t)cgc * ld);
  }
  const quat xa = qload(M + rac + (size_t)c * ld);
  // x at this wave's 4 columns (the same address across the wave: one fetch each)
  quat xc[SCW];
#pragma unroll
  for (int cc = 0; cc < SCW; ++cc) xc[cc] = qload(M + min(C0 + SCW * w + cc, n - 1) + (size_t)c * ld);
  const quat ua = (ra < n) ? xa : qzero();
  double qfl = 0.0;   // this thread's share of x^* M x over the tile
  // BF (the wide tiles): branch-free over the tile -- selects instead of
  // divergent ifs, and an inactive tile computes zeros from its clamped loads
  // and stores nothing -- so the body is one scheduling region: the
  // wave-uniform loads of x at the tile's columns issue alongside the tile
  // loads instead of after their wait, and the kernel needs 66 VGPRs instead
  // of 84 (three 512-thread blocks per CU instead of two).  2n = 8192 solve
  // -1.5 ms.  (Four blocks need 64: held to that it spills 20 bytes and the solve
  // takes 9 ms more, and with multiplies and adds for the quaternion product's
  // FMAs, which fits, it is slower too.)  The narrow tiles keep the branches: branch-free they made the
  // 512-problem batch 1.3% slower (also when held to five blocks per CU, their
  // residency with branches), for 0.7% on single solves of 2n <= 1024.
  constexpr bool BF = SW == 32;
  if (BF || active) {
    const double nua = BF ? qnorm2(ua) : 0.0;
    quat acc = qzero();
    double col[4 * SCW];
#pragma unroll
    for (int cc = 0; cc < SCW; ++cc) {
      const int cl = SCW * w + cc;
      const int cg = C0 + cl;
      const bool in = cg < n && ra < n && ra >= cg;
      const bool dg = ra == cg;   // the diagonal: real, enters x^* M x once (below twice)
      quat a, cp = qzero();
      if constexpr (BF) {
        a = quat{in ? qa[cc].ar : 0.0, (in && !dg) ? qa[cc].ai : 0.0, (in && !dg) ? qa[cc].br : 0.0,
                 (in && !dg) ? qa[cc].bi : 0.0};
        qfl = dg ? fma(-a.ar, nua, qfl) : qfl;
        qfma(acc, a, xc[cc]);   // a = 0 where cg >= n
        qfma_cl(cp, a, ua);
        const bool below = ra > cg;
        cp = quat{below ? cp.ar : 0.0, below ? cp.ai : 0.0, below ? cp.br : 0.0, below ? cp.bi : 0.0};
      } else {
        a = (cg < n && ra < n && ra >= cg) ? qa[cc] : qzero();
        if (ra == cg) {
          a = quat{a.ar, 0.0, 0.0, 0.0};
          qfl = fma(-a.ar, qnorm2(ua), qfl);
        }
        qfma(acc, a, cg < n ? xc[cc] : qzero());
        if (ra > cg) qfma_cl(cp, a, ua);
      }
      col[4 * cc + 0] = cp.ar; col[4 * cc + 1] = cp.ai; col[4 * cc + 2] = cp.br; col[4 * cc + 3] = cp.bi;
    }
    red[w][0][lane] = acc.ar;
    red[w][1][lane] = acc.ai;
    red[w][2][lane] = acc.br;
    red[w][3][lane] = acc.bi;
    // x^* M x over the tile's lower part, doubled off the diagonal: 2 Re(conj(x_i) acc_i)
    qfl = fma(2.0, qdot(ua, acc), qfl);
    // lane l ends with value vi = l / LPV (component vi & 3 of column vi >> 2), summed over the wave
    constexpr int LPV = 64 / (4 * SCW);
    const double cs = butterfly_sum<4 * SCW>(col);
    if (active && lane % LPV == 0) {
      const int vi = lane / LPV;
      const int cg = C0 + SCW * w + (vi >> 2);
      if (cg < n) reinterpret_cast<double*>(Pcol + (size_t)g * ldp + cg)[vi & 3] = cs;
    }
  }
  qfl = wave_sum_d(qfl);
  if (lane == 0) sqf[w] = qfl;
  __syncthreads();
  // wave v < 4 sums component v of the rows; the last wave x^* M x too
  if (tid == SYT - 64) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < SYT / 64; ++k) t += sqf[k];
    QF[b] = t;
  }
  if (active && w < 4) {
    const int i = R0 + lane;
    if (i < n && i >= C0) {
      double t = red[0][w][lane];
#pragma unroll
      for (int k = 1; k < NWV; ++k) t += red[k][w][lane];
      reinterpret_cast<double*>(Prow + (size_t)J * ldp + i)[w] = t;
    }
  }
}

// The arithmetic that finishes a column (k_wcol).  Every rounding is written
// out (explicit FMAs, no contraction of the rest), so that the variants of the
// kernel -- a solve and the batch it is a member of may run different ones --
// give the same bits.
//
// With x the raw column c, u = gamma x + delta e_1 (delta = u1 - gamma x1, row
// s0 = c + 1) and the panel's earlier columns V, W:
//   p   = y - V (W^* u) - W (V^* u),  y = M u = gamma (M x) + M[:, s0] delta
//         with (M x) from the matvec partials;
//   K   = u^* p / 2 = (u^* y - 2 Re(a^* b)) / 2,  a = W^* u, b = V^* u, and
//         u^* y = gamma^2 x^* M x + 2 gamma Re(conj(delta) (M x)_{s0}) + M_{s0 s0} |delta|^2,
//         x^* M x from the matvec's per-tile partials (QF) -- so every block
//         has K without a grid-wide reduction of p;
//   w_j = p - K u.
// Inside a panel, column c+1's pending update follows: subtract the
// [V W] [W V]^*-terms of the panel's columns 0..j, whose row-s0 coefficients
// (including the new w_j(s0) = p(s0) - K u1) every block forms redundantly.
// Row s0 itself is formed from these sums: u1, w_j(s0), and the diagonal
// entry d[c+1] of the updated column; the other rows start at s0 + 1, so that
// the 16-row groups of the tall-skinny partials are the rows of the next
// matvec's tiles.
//
// Block sums per column: qf = x^* M x, ab = Re(a^* b), wrow = (M x)_{s0},
// rd = V(s0,:) a + W(s0,:) b, cc = Re(V(s0,:) conj(W(s0,:))).
struct ColScalars {
  double gam, K;
  quat u1, delta, wc1;   // wc1 = w_j(s0)
  double dnext;          // the updated diagonal entry at s0
};
__device__ __forceinline__ ColScalars col_scalars(double qf, double ab, double cc, const quat& rd, const quat& wrow,
                                                  double gam, const quat& u1, const quat& x1, double m00) {
#pragma clang fp contract(off)
  ColScalars C;
  C.gam = gam;
  C.u1 = u1;
  C.delta = qaxpy(u1, -gam, x1);
  const double uy = fma(gam * gam, qf, fma(2.0 * gam, qdot(C.delta, wrow), m00 * qnorm2(C.delta)));
  C.K = 0.5 * fma(-2.0, ab, uy);
  const quat ps0 = qsub(qaxpy(qscale(wrow, gam), m00, C.delta), rd);
  C.wc1 = qaxpy(ps0, -C.K, u1);
  C.dnext = fma(-2.0, qdot(u1, C.wc1), fma(-2.0, cc, m00));
  return C;
}
// The block sums, each wave those whose terms it holds (about a third of the
// instructions per wave that one wave summing them all would take): wave 0 rd,
// wave 1 wrow, wave 2 ab and cc, all waves their terms of qf.
__device__ __forceinline__ void col_wave_sums(int wv, double qf, const quat& v4, double (*sh)[5]) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  if (wv < 3) {
    double v[4] = {v4.ar, v4.ai, v4.br, v4.bi};
    const double t = butterfly_sum<4>(v);
    if ((lane & 15) == 0) sh[wv][lane >> 4] = t;
  }
  qf = wave_sum_d(qf);
  if (lane == 0) sh[wv][4] = qf;
}
// One thread's share of a row, over the panel columns l = q + 16 k (its
// coefficients vv, ww): ps = gamma y - (V a + W b), us = V conj(W(s0)) + W
// conj(V(s0)); then summed over the wave's four q: lane 16 q' + r is left
// with components 2 q', 2 q' + 1 of row r's (ps, us), stored in red[r].
// RPAD: a row's 8 components and a gap of 2, which puts the 16 rows' 16-byte
// accesses in distinct banks.
constexpr int RPAD = 10;
template <int KPT>
__device__ __forceinline__ void row_share(const quat* vv, const quat* ww, const quat& yi, double gam, int q, int j,
                                          const quat* a, const quat* b, const quat* cw, const quat* cv,
                                          double (*red)[RPAD]) {
#pragma clang fp contract(off)
  quat accp = qscale(yi, gam), accu = qzero();
  // the coefficients beyond j are zero in LDS (and vv, ww finite), so no lane
  // masks are needed; a panel's first column has no terms
  if (j > 0)
#pragma unroll
    for (int k = 0; k < KPT; ++k) {
      const int l = q + 16 * k;
      const quat ak = a[l], bk = b[l], cwk = cw[l], cvk = cv[l];
      qfma(accp, qneg(vv[k]), ak);
      qfma(accp, qneg(ww[k]), bk);
      qfma(accu, vv[k], cwk);
      qfma(accu, ww[k], cvk);
    }
  double v[8] = {accp.ar, accp.ai, accp.br, accp.bi, accu.ar, accu.ai, accu.br, accu.bi};
  const int lane = threadIdx.x & 63;
  bstep<32, 4>(v, lane);
  bstep<16, 2>(v, lane);
  *reinterpret_cast<double2*>(&red[lane & 15][2 * (lane >> 4)]) = make_double2(v[0], v[1]);
}
// The row's results from the four waves' partials (red: wave, row, component):
// u, w_j and the updated entry of column c+1 (xi: x, ms: stale column s0).
struct RowOut {
  quat u, w, x;
};
__device__ __forceinline__ RowOut row_finish(const double (*red)[RQ][RPAD], int r, const ColScalars& C, const quat& xi,
                                             const quat& ms) {
#pragma clang fp contract(off)
  double t[8];
#pragma unroll
  for (int h = 0; h < 8; h += 2) {
    double2 s = *reinterpret_cast<const double2*>(&red[0][r][h]);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      const double2 z = *reinterpret_cast<const double2*>(&red[k][r][h]);
      s.x += z.x;
      s.y += z.y;
    }
    t[h] = s.x;
    t[h + 1] = s.y;
  }
  RowOut o;
  quat p = quat{t[0], t[1], t[2], t[3]};
  qfma(p, ms, C.delta);
  o.u = qscale(xi, C.gam);
  o.w = qaxpy(p, -C.K, o.u);
  o.x = qsub(ms, quat{t[4], t[5], t[6], t[7]});
  qfma_cr(o.x, qneg(o.u), C.wc1);
  qfma_cr(o.x, qneg(o.w), C.u1);
  return o;
}
// Tall-skinny partials of the updated column over the panel columns 0..j:
// this thread's columns l = q + 16 k (l = j: the new u, w) against x, summed
// over the 16 rows, to tsp[8 l + component] (W^* x, then V^* x).
template <int KPT>
__device__ __forceinline__ void row_tsp(const quat* vv, const quat* ww, const quat& u, const quat& w, const quat& x,
                                        int q, int j, double* tsp) {
#pragma clang fp contract(off)
  constexpr int NV = 8 * KPT;
  double v[NV];
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int l = q + 16 * k;
    quat ta = qzero(), tb = qzero();
    if (l <= j) {
      qfma_cl(ta, l == j ? w : ww[k], x);
      qfma_cl(tb, l == j ? u : vv[k], x);
    }
    v[8 * k + 0] = ta.ar; v[8 * k + 1] = ta.ai; v[8 * k + 2] = ta.br; v[8 * k + 3] = ta.bi;
    v[8 * k + 4] = tb.ar; v[8 * k + 5] = tb.ai; v[8 * k + 6] = tb.br; v[8 * k + 7] = tb.bi;
  }
  row16_halving<NV>(v);
  const int r = threadIdx.x & (RQ - 1);
  if constexpr (KPT == 1) {   // lane r holds value r / 2
    if ((r & 1) == 0 && q <= j) tsp[8 * q + (r >> 1)] = v[0];
  } else {
#pragma unroll
    for (int t = 0; t < NV / 16; ++t) {
      const int idx = r * (NV / 16) + t;
      const int l = q + 16 * (idx >> 3);
      if (l <= j) tsp[8 * l + (idx & 7)] = v[t];
    }
  }
}

// Column c's w_j and, inside a panel, column c+1's pending update, in one
// pass over rows s0 + 1 .. n - 1 (s0 = c + 1; 16 threads per row, KPT panel
// columns each): w_j stored in W[:, j], u in M[s0:, c], and unless column c
// closes its panel (j = nb - 1) or the reduction (c = n - 2) the updated
// column c+1 in M, its tail-norm partials in part, and the per-16-row partials
// of W^* x, V^* x in TSP.  Two barriers: the block sums, and the four waves'
// shares of each row; every thread then forms its row's results itself.
// At trailing sizes below ~1500 a block's time is one round trip to memory
// plus the instructions of one wave per SIMD, so both the barriers and the
// instruction count are its cost: two barriers instead of four, the eleven
// block sums by halving butterflies, each wave only those whose terms it holds,
// the sums in scalar registers, the row partials padded to distinct LDS banks,
// unconditional loads at clamped addresses, the batch addressing compiled out
// of single solves.  Per column with its matvec at panel width 16: 9.8 us ->
// 8.2 us; 2n = 1024 reduction 4.74 -> 4.07 ms, 2n = 8192 111.0 -> 104.3 ms.
// Fusing it into the next column's matvec (one launch per column, every tile
// block repeating the row work of its 96 rows) took 11-12 us
// per column: twice the instructions on every wave.
// PY, PQ: partial loads per thread per gather batch (quaternion row partials,
// x^* M x partials); WPE: the waves per SIMD the register budget aims at.
template <int KPT, int PY, int PQ, int WPE, bool BT>
__global__ void __launch_bounds__(RB) __attribute__((amdgpu_waves_per_eu(WPE))) k_wcol(
    quat* __restrict__ M, quat* __restrict__ W, const quat* __restrict__ Prow, int pcs, int ld,
    int n, int p, int c, int j, int ldw, int ldp, int nb, const quat* __restrict__ TS, const double* __restrict__ scal,
    const double* __restrict__ QF, double* __restrict__ part, double* __restrict__ TSP, double* __restrict__ d,
    int ldtsp, int tsm, ZB zb) {
  int bx = blockIdx.x;
  if constexpr (BT) {
    int z;
    if (!fold_member(zb, [=](int m) { return wcol_blocks(m - c - 1); }, z, n, bx)) return;
    M = zoff(M, zb, z); W = zoff(W, zb, z); Prow = zoff(Prow, zb, z); TS = zoff(TS, zb, z);
    scal = zoff(scal, zb, z); QF = zoff(QF, zb, z); part = zoff(part, zb, z); TSP = zoff(TSP, zb, z); d = zoff(d, zb, z);
  }
  __shared__ quat a[NBMAX], b[NBMAX], cw[NBMAX], cv[NBMAX];
  __shared__ __align__(16) double red[RB / 64][RQ][RPAD];   // wave, row, (p | column update) component
  __shared__ double shr[RB / 64][5];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s0 = c + 1;
  const bool more = (j + 1 < nb) && (c + 1 <= n - 2);   // uniform
  const int r = tid & (RQ - 1), q = tid >> 4;
  const int i = s0 + 1 + bx * RQ + r;
  const int ic = min(i, n - 1);
  const int jl = j > 0 ? j - 1 : 0;
  // ---- loads, all issued up front
  quat vv[KPT], ww[KPT];
#pragma unroll
  for (int k = 0; k < KPT; ++k) {
    const int l = min(q + 16 * k, jl);
    vv[k] = qload(M + ic + (size_t)(p + l) * ld);
    ww[k] = qload(W + ic + (size_t)l * ldw);
  }
  const quat xi = qload(M + ic + (size_t)c * ld);
  const quat ms = qload(M + ic + (size_t)s0 * ld);   // stale column s0 = c+1 (row i)
  // The column scalars (gamma, u1, x1, M[s0, s0]) in one vector load over
  // lanes 0..9, taken apart after the partial gathers.  As scalar loads they
  // would share the scalar-load counter with the kernel arguments the gather
  // loop needs, and the loop's loads could not issue before they arrived.
  const double sv = scal[min(lane, 9)];
  // waves 0 and 2: the panel's coefficients, lane l those of columns l + 64 h
  constexpr int NH = (16 * KPT + 63) / 64;
  quat al[NH], bl[NH], cwl[NH], cvl[NH];
  if ((wv & 1) == 0)
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      al[h] = bl[h] = cwl[h] = cvl[h] = qzero();
      const int l = lane + 64 * h;
      if (l < j) {
        al[h] = qload(TS + l);
        bl[h] = qload(TS + nb + l);
        cwl[h] = qload(W + s0 + (size_t)l * ldw);
        cvl[h] = qload(M + s0 + (size_t)(p + l) * ld);
      }
    }
  const int G = (n - s0 + SG - 1) / SG;
  // The matvec partials this thread sums, gathered in fixed-size batches at
  // clamped addresses (surplus values are dropped), so that one wait covers
  // them all (one batch up to trailing sizes of ~4k rows with the wide variant,
  // ~1k with the light one) and no load sits in a branch of its own:
  //   y(i):  slots k = q + 16 t of row i's list, Prow[J][i] for J <= li / SW
  //          (SW the strip width of this trailing size)
  //          (k < nJ), then Pcol[g][i] for g >= li / SG (slot pcs + g of Prow);
  //   x^* M x: QF[tid + RB t], t over the G (G + 1) tile partials;
  //   (M x)_{s0}: Prow[0][s0] and Pcol[g][s0] as slots lane + 64 t of G + 1, in wave 1.
  const int li = ic - s0;
  const int spg = matvec_spg(n - s0, tsm);
  const int nJ = (spg == 4 ? li >> 4 : li >> 5) + 1, g0 = li / SG;
  const int ns = nJ + G - g0;   // slots of row i
  const int shift = pcs + g0 - nJ;
  const int cy = cdiv_d(ns - q, 16);
  const int nq = ntiles(G, spg);
  const int cq = cdiv_d(nq - tid, RB);
  const int cw0 = wv == 1 ? cdiv_d(G + 1 - lane, 64) : 0;
  quat yi = qzero(), w0 = qzero();
  double qf = 0.0;
  // surplus values are dropped by a factor 0: one select where zeroing the
  // value takes eight (they repeat the row's last slot, so a NaN or infinity
  // there is in the row's sum anyway)
  auto gather = [&](int bt) {
    quat py[PY];
    double pq[PQ];
#pragma unroll
    for (int u = 0; u < PY; ++u) {
      const int k = min(q + 16 * (bt * PY + u), ns - 1);
      py[u] = qload(Prow + (unsigned)((k < nJ ? k : k + shift) * ldp + ic));
    }
#pragma unroll
    for (int u = 0; u < PQ; ++u) pq[u] = QF[(unsigned)min(tid + RB * (bt * PQ + u), nq - 1)];
    quat pw;
    if (wv == 1) {
      const int k = min(lane + 64 * bt, G);
      pw = qload(Prow + (unsigned)((k == 0 ? 0 : pcs + k - 1) * ldp + s0));
    }
#pragma unroll
    for (int u = 0; u < PY; ++u) yi = qaxpy(yi, bt * PY + u < cy ? 1.0 : 0.0, py[u]);
#pragma unroll
    for (int u = 0; u < PQ; ++u) qf = fma(bt * PQ + u < cq ? 1.0 : 0.0, pq[u], qf);
    if (wv == 1) w0 = qaxpy(w0, bt < cw0 ? 1.0 : 0.0, pw);
  };
  gather(0);
  const int nbt = max(max(cdiv_d(ns, 16 * PY), cdiv_d(nq, RB * PQ)), cdiv_d(G + 1, 64));
  for (int bt = 1; bt < nbt; ++bt) gather(bt);
  {
#pragma clang fp contract(off)
    quat v4 = w0;
    if (wv == 0) {
      v4 = qzero();
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        qfma(v4, cvl[h], al[h]);
        qfma(v4, cwl[h], bl[h]);
      }
    } else if (wv == 2) {
      v4 = qzero();
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        v4.ar += qdot(al[h], bl[h]);
        v4.ai += qdot(cvl[h], cwl[h]);
        const int l = lane + 64 * h;
        if (l < 16 * KPT) {   // zero beyond j
          a[l] = al[h];
          b[l] = bl[h];
          cw[l] = qconj(cwl[h]);
          cv[l] = qconj(cvl[h]);
        }
      }
    }
    col_wave_sums(wv, qf, v4, shr);
  }
  __syncthreads();
  // lane 5 w + t holds sum t of wave w; to scalar registers
  const double st = (&shr[0][0])[min(lane, 19)];
  const double qs = ((lane_d(st, 4) + lane_d(st, 9)) + lane_d(st, 14)) + lane_d(st, 19);
  const ColScalars C = col_scalars(qs, lane_d(st, 10), lane_d(st, 11),
                                   quat{lane_d(st, 0), lane_d(st, 1), lane_d(st, 2), lane_d(st, 3)},
                                   quat{lane_d(st, 5), lane_d(st, 6), lane_d(st, 7), lane_d(st, 8)}, lane_d(sv, 0),
                                   quat{lane_d(sv, 1), lane_d(sv, 2), lane_d(sv, 3), lane_d(sv, 4)},
                                   quat{lane_d(sv, 5), lane_d(sv, 6), lane_d(sv, 7), lane_d(sv, 8)}, lane_d(sv, 9));
  if (bx == 0 && tid == 0) {   // row s0
    qstore(M + s0 + (size_t)c * ld, C.u1);
    qstore(W + s0 + (size_t)j * ldw, C.wc1);
    if (more) d[s0] = C.dnext;
  }
  row_share<KPT>(vv, ww, yi, C.gam, q, j, a, b, cw, cv, red[wv]);
  __syncthreads();
  RowOut o = row_finish(red, r, C, xi, ms);
  // every wave has every row's results (in its lanes 0..15): one store each
  if (lane < RQ && i < n) {
    if (wv == 0) qstore(W + i + (size_t)j * ldw, o.w);
    else if (wv == 1) qstore(M + i + (size_t)c * ld, o.u);
    else if (wv == 2 && more) qstore(M + i + (size_t)s0 * ld, o.x);
  }
  if (!more) return;   // uniform
  // row s0 + 1 is the updated column's x_1: not in its tail
  if (i <= s0 + 1 || i >= n) o.x = qzero();
  if (wv == 3) {
    double ss = qnorm2(o.x);   // lanes 0..15: the 16 rows
    ss += xlane<1>(ss);
    ss += xlane<2>(ss);
    ss += xlane<4>(ss);
    ss += xlane<8>(ss);
    if (lane == 0) part[bx] = ss;
  }
  row_tsp<KPT>(vv, ww, o.u, o.w, o.x, q, j, TSP + (size_t)bx * ldtsp);
}

// ---------------------------------------------------------------------------
// Register-resident tail.  Once the trailing matrix has at most TAILN rows,
// one workgroup per problem finishes the reduction: per column the reflector,
// y = A u, K = u^* y / 2, w = y - K u and the rank-2 update A -= u w^* + w u^*
// at once (unblocked: no panel, no W), separated by barriers instead of kernel
// launches.  It starts at a panel boundary p, after the trailing update of the
// panel before it, and writes d and e of columns p .. n-2, d[n-1], and the
// reflectors u into M below the subdiagonal (the blocked columns'
// conventions).
//
// The whole Hermitian block (both triangles) is held in registers: lane = row,
// and wave v owns columns v, v + 8, ... (cyclic, so that the waves stay
// evenly loaded as columns retire).  The matrix is never re-read: per
// column only u, w (broadcast reads) and the waves' partials of y pass
// through LDS, with three barriers.  Wave cl % 8 owns column cl, so after the
// update of column cl - 1 it forms the next reflector from its own registers
// while the other waves are still updating.  Retired and absent rows and
// columns have u = w = 0, so no lane masks are needed.  A version with the
// block in LDS and four waves was bound by its re-reads of the block, one wave
// per SIMD having nothing to hide them behind: 64 columns took 242 us, now
// 138 us (149 with 16 waves, 140 with 4; 149 with the stages in one rolled
// loop, although that quarters the code).  Two blocks fit a CU at up to 128
// registers: with one (136) a batch of 2048 of 2n = 32 .. 64 takes 1.54 ms, with
// two 1.37.
// Waves pass over absent columns: with their zeros multiplied too,
// eigenvalues only of 2n = 32 took 99 us where the LDS form took 90; now 80 (2n = 64
// 145 -> 119.5 us, 112 201 -> 190, 128 216.0 -> 216.8).
// ---------------------------------------------------------------------------
constexpr int TT = 512;            // threads: 8 waves
constexpr int TWV = TT / 64;
constexpr int TKC = TAILN / TWV;    // columns per wave
static_assert(TAILN == 64 && TKC * TWV == TAILN, "k_tail: lane = row, TKC columns per wave");

__global__ void __launch_bounds__(TT, 4) k_tail(quat* __restrict__ M, int ld, int n, int p,
                                  const int* __restrict__ pstart,
                                             double* __restrict__ d, quat* __restrict__ e, ZB zb) {
  if (zb.nvec) {
    n = zb.nvec[blockIdx.z];
    p = pstart[blockIdx.z];
    M = zoff(M, zb); d = zoff(d, zb); e = zoff(e, zb);
  }
  const int ms = n - p;
  if (ms < 1 || ms > TAILN) return;   // uniform: a problem without a tail
  __shared__ quat us[2][TAILN], ys[2][TAILN];   // u and w, by column parity
  __shared__ quat part[TWV][TAILN];             // the waves' partials of A u
  const int tx = threadIdx.x & 63;              // row
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  quat a[TKC];   // elements (tx, wv + TWV k)
#pragma unroll
  for (int k = 0; k < TKC; ++k) {
    const int j = wv + TWV * k;
    a[k] = qzero();
    if (tx < ms && j < ms) {
      a[k] = tx >= j ? qload(M + (p + tx) + (size_t)(p + j) * ld) : qconj(qload(M + (p + j) + (size_t)(p + tx) * ld));
      if (tx == j) a[k] = quat{a[k].ar, 0.0, 0.0, 0.0};
    }
  }
  // The reflector of column cl from its owner's registers (column x).  A block
  // may shrink by a roundoff per column (equal entries: what is left of each
  // column is the rounding of equal sums), down to where squares lose digits and
  // u^* u is no longer 2; there the column is scaled up first.
  auto reflect = [&](int cl, const quat& x) {
    const int r0 = cl + 1;
    const bool row = tx >= r0 && tx < ms;
    double tail = wave_sum_d(tx > r0 && tx < ms ? qnorm2(x) : 0.0);
    quat x1 = quat{lane_d(x.ar, r0), lane_d(x.ai, r0), lane_d(x.br, r0), lane_d(x.bi, r0)};
    double up = 1.0;
    if (qnorm2(x1) + tail < TINY_SQ) {   // uniform
      up = UPSCALE;
      tail = wave_sum_d(tx > r0 && tx < ms ? qnorm2(qscale(x, up)) : 0.0);
      x1 = qscale(x1, up);
    }
    quat alpha;
    const Refl R = reflector(x1, tail, &alpha);
    if (tx == cl) {
      d[p + cl] = x.ar;
      qstore(e + p + cl, qscale(alpha, up == 1.0 ? 1.0 : 1.0 / UPSCALE));
    }
    const quat ui = row ? (tx == r0 ? R.u1 : qscale(qscale(x, up), R.g)) : qzero();
    us[cl & 1][tx] = ui;
    if (row) qstore(M + (p + tx) + (size_t)(p + cl) * ld, ui);
  };
  if (wv == 0 && ms > 1) reflect(0, a[0]);
#pragma unroll
  for (int kk = 0; kk < TKC; ++kk) {
    for (int c = 0; c < TWV; ++c) {
      const int cl = TWV * kk + c;
      if (cl + 1 >= ms) break;   // uniform
      const int r0 = cl + 1, par = cl & 1;
      const unsigned nt = ms - r0;   // trailing rows
      __syncthreads();   // us of column cl is complete
      const quat ui = us[par][tx];
      quat acc = qzero();   // this lane's row of A u over this wave's columns
#pragma unroll
      for (int k = kk; k < TKC; ++k)
        if (unsigned(wv + TWV * k - r0) < nt) qfma(acc, a[k], us[par][wv + TWV * k]);   // uniform: r0 .. ms - 1
      part[wv][tx] = acc;
      __syncthreads();
      if (wv == 0) {
        quat y = part[0][tx];
#pragma unroll
        for (int k = 1; k < TWV; ++k) y = qadd(y, part[k][tx]);
        // K = u^* y / 2; u = 0 outside the trailing rows
        const double K = 0.5 * wave_sum_d(ui.ar * y.ar + ui.ai * y.ai + ui.br * y.br + ui.bi * y.bi);
        ys[par][tx] = (tx >= r0 && tx < ms) ? qsub(y, qscale(ui, K)) : qzero();   // w
      }
      __syncthreads();
      const quat wi = ys[par][tx];
      // the rank-2 update; the wave owning the next column forms its
      // reflector right after updating that column, before its others
#pragma unroll
      for (int k = kk; k < TKC; ++k) {
        const int j = wv + TWV * k;
        if (unsigned(j - r0) >= nt) continue;   // uniform
        const quat uj = us[par][j], wj = ys[par][j];
        const quat nu = quat{-ui.ar, -ui.ai, -ui.br, -ui.bi}, nw = quat{-wi.ar, -wi.ai, -wi.br, -wi.bi};
        qfma_cr(a[k], nu, wj);
        qfma_cr(a[k], nw, uj);
        if (tx == j) a[k] = quat{a[k].ar, 0.0, 0.0, 0.0};   // Hermitian diagonal: real
        if (j == r0 && r0 + 1 < ms) reflect(r0, a[k]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < TKC; ++k)
    if (wv + TWV * k == ms - 1 && tx == ms - 1) d[n - 1] = a[k].ar;
}

int tail_start(int n, int nb) {
  if (n <= TAILN) return 0;
  const int p = (n - TAILN + nb - 1) / nb * nb;
  return p <= n - 1 ? p : n;
}

__global__ void k_last_diag(const quat* __restrict__ M, int ld, int n, double* __restrict__ d, ZB zb) {
  if (zb.nvec) {
    n = zb.nvec[blockIdx.z];
    M = zoff(M, zb); d = zoff(d, zb);
  }
  if (threadIdx.x == 0) d[n - 1] = M[(n - 1) + (size_t)(n - 1) * ld].ar;
}

static inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// (sized for any switch up to TSM_MAX)
int matvec_row_slots(int nmax) { return std::max(cdiv(nmax, 32), cdiv(std::min(nmax, TSM_MAX), 16)); }
int matvec_col_slots(int nmax) { return (nmax + SG - 1) / SG; }
int matvec_tile_slots(int nmax) {
  return std::max(ntiles(cdiv(nmax, SG) + 1, 2), ntiles(cdiv(std::min(nmax, TSM_MAX), SG) + 1, 4));
}

// panel columns per thread (16 threads per row) as a compile-time bound
static int kpt_for(int nb) {
  const int k = cdiv(nb, 16);
  return k <= 1 ? 1 : k <= 2 ? 2 : k <= 4 ? 4 : 8;
}

// k_wcol variants: light gathers (more blocks per CU: batches of small
// problems) up to trailing size 1536, wide ones (one gather batch) above.
template <int KPT, bool BT, class... Args>
static void launch_wcol_k(int sz, dim3 grid, hipStream_t s, Args... args) {
  // register budgets that compile without spills: 3 waves per SIMD at KPT 1,
  // 2 at KPT 2 and 4, 1 at KPT 8
  constexpr int WPE = KPT == 1 ? 3 : (KPT == 8 ? 1 : 2);
  if (sz <= 1536) hipLaunchKernelGGL((k_wcol<KPT, 4, 2, WPE, BT>), grid, dim3(RB), 0, s, args...);
  else hipLaunchKernelGGL((k_wcol<KPT, 10, 18, 1, BT>), grid, dim3(RB), 0, s, args...);
}
template <bool BT, class... Args>
static void launch_wcol(int kpt, int sz, dim3 grid, hipStream_t s, Args... args) {
  switch (kpt) {
    case 1: launch_wcol_k<1, BT>(sz, grid, s, args...); break;
    case 2: launch_wcol_k<2, BT>(sz, grid, s, args...); break;
    case 4: launch_wcol_k<4, BT>(sz, grid, s, args...); break;
    default: launch_wcol_k<8, BT>(sz, grid, s, args...); break;
  }
}

// Per panel: per column k_symv and k_wcol (which also updates the next
// column of the panel and leaves its tail-norm partials); then the trailing
// update.
int reduce(quat* M, int n, int ld, int nb, double* d, quat* e, const ReduceWork& w, hipStream_t s) {
  if (n <= 0) return ZQI_OK;
  if (nb < 1 || nb > NBMAX || w.tsm < 0 || w.tsm > TSM_MAX) return ZQI_ERR_ARG;
  if (n == 1) {
    hipLaunchKernelGGL(k_last_diag, dim3(1), dim3(64), 0, s, M, ld, n, d, ZB{nullptr, 0});
    return hipGetLastError() == hipSuccess ? ZQI_OK : ZQI_ERR_HIP;
  }
  const int ldw = n;
  const int kpt = kpt_for(nb);
  const int ts = tail_start(n, nb);   // n: no tail
  for (int p = 0; p < n - 1 && p < ts; p += nb) {
    const int wdt = (nb < n - 1 - p) ? nb : (n - 1 - p);
    for (int j = 0; j < wdt; ++j) {
      const int c = p + j;
      const int sz = n - c - 1;                    // trailing size
      const int nparts = cdiv(sz, RQ);             // partials the column kernel left for this column
      const int G = cdiv(sz, SG);
      const int spg = matvec_spg(sz, w.tsm);
      const int nmain = ntiles(G, spg) + (j > 0 ? (8 * j + 63) / 64 : 1);
      {
        // algorithmic bytes: one read of the trailing lower triangle
        ProfScope ps(PROF_SYMV, s, 32.0 * 0.5 * (double)sz * (sz + 1));
        if (spg == 4)
          launch_k(k_symv<256, 16, false>, dim3(nmain), dim3(256), 0, s, M, w.W, w.TSP, w.part, ld, n, p, c, j, ldw,
                   nparts, w.ldtsp, w.scal, d, e, w.Prow, w.Pcol, n, nb, w.TS, w.QF, ZB{nullptr, 0});
        else
          launch_k(k_symv<512, 32, false>, dim3(nmain), dim3(512), 0, s, M, w.W, w.TSP, w.part, ld, n, p, c, j, ldw,
                   nparts, w.ldtsp, w.scal, d, e, w.Prow, w.Pcol, n, nb, w.TS, w.QF, ZB{nullptr, 0});
      }
      launch_wcol<false>(kpt, sz, dim3(wcol_blocks(sz)), s, M, w.W, w.Prow, w.pcs, ld, n, p, c, j, ldw,
                         n, nb, w.TS, w.scal, w.QF, w.part, w.TSP, d, w.ldtsp, w.tsm, ZB{nullptr, 0});
    }
    // trailing update of rows/cols [p+wdt, n): M -= [V W] [W V]^*  (lower triangle)
    const int r0 = p + wdt;
    const int mt = n - r0;
    if (mt > 0) {
      QOperand A{M + r0 + (size_t)p * ld, w.W + r0, ld, ldw, wdt, false, INT_MIN / 2};
      QOperand B{w.W + r0, M + r0 + (size_t)p * ld, ldw, ld, wdt, true, INT_MIN / 2};
      // algorithmic flops: lower triangle x rank 2*wdt, 32 flops per quaternion multiply-add
      ProfScope ps(PROF_TRAIL, s, 32.0 * 0.5 * (double)mt * (mt + 1) * 2.0 * wdt);
      int rc = qgemm(mt, mt, 2 * wdt, -1.0, A, B, 1.0, M + r0 + (size_t)r0 * ld, ld, true, s);
      if (rc) return rc;
    }
  }
  if (ts < n) hipLaunchKernelGGL(k_tail, dim3(1), dim3(TT), 0, s, M, ld, n, ts, nullptr, d, e, ZB{nullptr, 0});
  else hipLaunchKernelGGL(k_last_diag, dim3(1), dim3(64), 0, s, M, ld, n, d, ZB{nullptr, 0});
  return hipGetLastError() == hipSuccess ? ZQI_OK : ZQI_ERR_HIP;
}

// problem z's workspace: the batch base pointer advanced by z slabs
template <class T>
static T* zshift(T* p, size_t bytes) {
  using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return reinterpret_cast<T*>(reinterpret_cast<B*>(p) + bytes);
}

size_t reduce_batched_tasks(int nprob, const int* nh, int nb) {
  if (nprob <= 0 || nh[0] < 2) return 1;
  return (size_t)nprob * cdiv(nh[0] - 1, nb) + 1;
}

int reduce_batched(int nprob, const int* nh, ZB zb, quat* M, int ld, int nb, double* d, quat* e, const ReduceWork& w,
                   QGemmTask* tasks, int* tstart, Staging& st, hipStream_t s) {
  if (nprob <= 0) return ZQI_OK;
  if (nb < 1 || nb > NBMAX || w.tsm < 0 || w.tsm > TSM_MAX) return ZQI_ERR_ARG;
  const int L = nh[0];
  for (int z = 1; z < nprob; ++z)
    if (nh[z] > nh[z - 1] || nh[z] < 1) return ZQI_ERR_ARG;
  const int ldw = ld;
  // problem z runs the blocked columns c < lim[z] in lockstep and its tail
  // (k_tail) from ts[z]; both are non-increasing in z (sizes descending)
  std::vector<int> ts(nprob), lim(nprob);
  for (int z = 0; z < nprob; ++z) {
    ts[z] = tail_start(nh[z], nb);
    lim[z] = std::min(ts[z], nh[z] - 1);
  }
  const int npan = L > 1 ? cdiv(L - 1, nb) : 0;
  // trailing-update tasks of every panel, problem by problem: the task of
  // problem z in panel P is what reduce() launches for z after that panel
  std::vector<QGemmTask> tt;
  std::vector<int> toff(npan + 1, 0), tmaxm(npan, 0);
  std::vector<double> tflops(npan, 0.0);   // algorithmic flops of each panel's trailing updates
  for (int P = 0; P < npan; ++P) {
    const int p = P * nb;
    toff[P] = (int)tt.size();
    for (int z = 0; z < nprob && nh[z] - 1 > p; ++z) {
      if (p >= ts[z]) continue;
      const int n = nh[z];
      const int wdt = std::min(nb, n - 1 - p);
      const int r0 = p + wdt, mt = n - r0;
      if (mt <= 0) continue;
      quat* Mz = reinterpret_cast<quat*>(reinterpret_cast<char*>(M) + (size_t)z * zb.zs);
      quat* Wz = reinterpret_cast<quat*>(reinterpret_cast<char*>(w.W) + (size_t)z * zb.zs);
      QOperand A{Mz + r0 + (size_t)p * ld, Wz + r0, ld, ldw, wdt, false, INT_MIN / 2};
      QOperand B{Wz + r0, Mz + r0 + (size_t)p * ld, ldw, ld, wdt, true, INT_MIN / 2};
      tt.push_back(QGemmTask{mt, mt, 0, 2 * wdt, ld, 1, -1.0, 1.0, A, B, Mz + r0 + (size_t)r0 * ld});
      tmaxm[P] = std::max(tmaxm[P], mt);
      tflops[P] += 32.0 * 0.5 * (double)mt * (mt + 1) * 2.0 * wdt;
    }
  }
  toff[npan] = (int)tt.size();
  if (tt.size() > reduce_batched_tasks(nprob, nh, nb)) return ZQI_ERR_ARG;
  int rc = stage_upload(st, tt.data(), tt.size() * sizeof(QGemmTask), tasks, s);
  if (rc) return rc;
  if ((rc = stage_upload(st, ts.data(), nprob * sizeof(int), tstart, s))) return rc;
  const int kpt = kpt_for(nb);
  const int cend = lim[0];
  int act = nprob;   // problems with a blocked column c: c < lim[z] (a prefix)
  for (int c = 0; c < cend; ++c) {
    while (act > 0 && lim[act - 1] <= c) --act;
    const int p = (c / nb) * nb, j = c - p;
    const int sz = L - c - 1;
    const int nparts = cdiv(sz, RQ);
    const int NF = j > 0 ? (8 * j + 63) / 64 : 1;
    // each problem's matvec takes the tile shape of its own trailing size:
    // problems [0, k1) wide strips, [k1, act) narrow ones (sizes descending)
    int k1 = 0;
    while (k1 < act && matvec_spg(nh[k1] - c - 1, w.tsm) == 2) ++k1;
    // algorithmic bytes of a launch: one read of each member's trailing lower triangle
    auto tri_bytes = [&](int z0, int z1) {
      double b = 0.0;
      for (int z = z0; z < z1; ++z) b += 32.0 * 0.5 * (double)(nh[z] - c - 1) * (nh[z] - c);
      return b;
    };
    if (k1 > 0) {
      ProfScope ps(PROF_SYMV, s, tri_bytes(0, k1));
      const int gx = fold_width(k1, [&](int z) { return symv_blocks(nh[z] - c - 1, 2, NF); });
      launch_k(k_symv<512, 32, true>, dim3(gx, 1, (k1 + 1) / 2), dim3(512), 0, s, M, w.W, w.TSP,
               w.part, ld, L, p, c, j, ldw, nparts, w.ldtsp, w.scal, d, e, w.Prow, w.Pcol, ld, nb, w.TS, w.QF,
               ZB{zb.nvec, zb.zs, k1});
    }
    if (k1 < act) {
      const size_t sh = (size_t)k1 * zb.zs;
      const int gx = fold_width(act - k1, [&](int z) { return symv_blocks(nh[k1 + z] - c - 1, 4, NF); });
      ProfScope ps(PROF_SYMV, s, tri_bytes(k1, act));
      launch_k(k_symv<256, 16, true>, dim3(gx, 1, (act - k1 + 1) / 2), dim3(256), 0, s, zshift(M,
               sh), zshift(w.W, sh), zshift(w.TSP, sh), zshift(w.part, sh), ld, L, p, c, j, ldw, nparts, w.ldtsp,
               zshift(w.scal, sh), zshift(d, sh), zshift(e, sh), zshift(w.Prow, sh), zshift(w.Pcol, sh), ld, nb,
               zshift(w.TS, sh), zshift(w.QF, sh), ZB{zb.nvec + k1, zb.zs, act - k1});
    }
    const int gw = fold_width(act, [&](int z) { return wcol_blocks(nh[z] - c - 1); });
    launch_wcol<true>(kpt, sz, dim3(gw, 1, (act + 1) / 2), s, M, w.W, w.Prow, w.pcs, ld, L, p, c, j,
                      ldw, ld, nb, w.TS, w.scal, w.QF, w.part, w.TSP, d, w.ldtsp, w.tsm,
                      ZB{zb.nvec, zb.zs, act});
    if (j == nb - 1 || c == cend - 1) {
      const int P = c / nb;
      const int cnt = toff[P + 1] - toff[P];
      ProfScope ps(PROF_TRAIL, s, tflops[P]);
      if (cnt > 0 && (rc = qgemm_tasks(tasks + toff[P], tt.data() + toff[P], cnt, tmaxm[P], tmaxm[P], 0, false, true,
                                       true, s)))
        return rc;
    }
  }
  // problems without a tail take d[n-1] here; the tails overwrite theirs
  hipLaunchKernelGGL(k_last_diag, dim3(1, 1, nprob), dim3(64), 0, s, M, ld, L, d, zb);
  hipLaunchKernelGGL(k_tail, dim3(1, 1, nprob), dim3(TT), 0, s, M, ld, L, 0, tstart, d, e, zb);
  return hipGetLastError() == hipSuccess ? ZQI_OK : ZQI_ERR_HIP;
}

}  // namespace zq
