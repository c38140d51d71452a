// Batched SVD of the block matrices of a block-sparse tensor, in FP64 and
// complex128, by one-sided block Jacobi.  It replaces MatSVD (framework/
// hp_numeric/lapack.h:41-82 gesvd, GPU :811-1011) called once per block matrix
// by DataBlkDecompSVD (qltensor/blk_spar_data_ten/data_blk_operations.h:
// 630-663); here every block matrix of the tensor is decomposed in one batched
// launch sequence.
//
// SVD.  The working matrix X is A (rows >= cols) or A^H (rows < cols), stored
// column-major so that columns are contiguous; V starts as the identity.  The
// columns are split into blocks of kB; every round of a sweep pairs the
// blocks by the circle method, and for every block pair
//   1. one workgroup per kRG-row group forms that group's part of the Gram
//      matrix G = P^H P of the panel P = [X_I X_J],
//   2. one workgroup sums the parts in group order, skips the pair when
//      max |G_pq| / sqrt(G_pp G_qq) < tol, and otherwise diagonalises G in
//      LDS by one sweep of cyclic two-sided Jacobi, accumulating the unitary
//      Q (G <- J^H G J, Q <- Q J per rotation; the outer sweeps repeat the
//      pair until its columns are orthogonal, so the solve need not finish),
//   3. one workgroup per kUR-row group updates P <- P Q and the matching
//      columns of V <- V Q.
// Spreading the rows over workgroups keeps the chip busy on the few large
// block matrices, whose pairs set the length of a round.
// Before every sweep the columns are ordered by decreasing norm (the block
// order follows it), which keeps graded spectra to a few sweeps.  A matrix
// whose sweep rotates nothing has converged; then sigma_j = |X_j|,
// U_j = X_j / sigma_j (zero when sigma_j = 0) and A = U diag(sigma) V^H,
// sorted by decreasing sigma (ties by column).

#include <algorithm>
#include <cmath>
#include <vector>

#include "block_dense.h"

using namespace qlt::dense;

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kSolveThreads = 512;   // of the Gram and solve workgroups
constexpr int kB = 16;          // columns per Jacobi block
constexpr int kW = 2 * kB;      // panel width
constexpr int kRG = 64;         // rows per Gram workgroup
constexpr int kUR = 32;         // rows per update workgroup
constexpr int kMaxSweeps = 40;
constexpr int kMaxSortCols = 4096;   // LDS bound of the per-matrix column sort

struct SvdMat {
  int64_t M, N;       // working shape (M >= N)
  int64_t x_off;      // X: column-major M x N, in elements of the workspace
  int64_t v_off;      // V: column-major N x N
  int64_t p_off;      // column order (int32), in int32 elements
  int64_t m, n;       // caller shape
  int64_t a_off, u_off, s_off, vt_off;
  int32_t nb, P;      // column blocks; players of the circle method (even)
  int32_t tr;         // X = A^H
  int32_t ng;         // row groups of X (kRG rows each)
  int32_t pair0;      // first pair slot of the matrix (P / 2 slots)
  int32_t pad;
  int64_t gram0;      // first partial-Gram slot (P / 2 * ng slots)
};

struct SvdItem {
  int32_t mat;
  int32_t k;          // pair index within a round
};

// One row group of one pair: rows g * kRG .. of X (phase 1), or g * kUR .. of X
// (kind 0) or V (kind 1; phase 3).
struct SvdRowItem {
  int32_t mat;
  int32_t k;
  int32_t g;
  int32_t kind;
};

// Circle-method pairing: `players` even, round r in [0, players - 1), pair
// k in [0, players / 2).  Both sums lie in [0, 2 (players - 1)), so one
// conditional subtraction reduces them modulo players - 1.
__device__ __forceinline__ void circle_pair(int players, int r, int k, int &a, int &b) {
  const int m = players - 1;
  const int x = r + k, y = r - k + m;
  a = k == 0 ? m : x >= m ? x - m : x;
  b = y >= m ? y - m : y;
}

// The arithmetic of a rotation, its fused multiply-adds written out: what the
// compiler fuses depends on the code around, and the phases of the singular
// vectors hang on the last bits of inner products that are only rounding.
__device__ __forceinline__ double sq_(double a) { return a * a; }
__device__ __forceinline__ double sq_(cplx a) { return fma(a.x, a.x, a.y * a.y); }
// e * b, and conj(e) * b
__device__ __forceinline__ double phase_(double e, double b) { return e * b; }
__device__ __forceinline__ cplx phase_(cplx e, cplx b) {
  return {fma(e.x, b.x, -(e.y * b.y)), fma(e.y, b.x, e.x * b.y)};
}
__device__ __forceinline__ double cphase_(double e, double b) { return e * b; }
__device__ __forceinline__ cplx cphase_(cplx e, cplx b) {
  return {fma(e.x, b.x, e.y * b.y), fma(e.x, b.y, -(e.y * b.x))};
}
// c a - s b, and s a + c b
__device__ __forceinline__ double rot_p(double c, double s, double a, double b) { return fma(c, a, -(s * b)); }
__device__ __forceinline__ cplx rot_p(double c, double s, cplx a, cplx b) {
  return {rot_p(c, s, a.x, b.x), rot_p(c, s, a.y, b.y)};
}
__device__ __forceinline__ double rot_q(double c, double s, double a, double b) { return fma(s, a, c * b); }
__device__ __forceinline__ cplx rot_q(double c, double s, cplx a, cplx b) {
  return {rot_q(c, s, a.x, b.x), rot_q(c, s, a.y, b.y)};
}

template <bool C>
__global__ void __launch_bounds__(kThreads) k_svd_load(const SvdMat *mats, const void *a_, void *ws_, int32_t *perm) {
  using T = typename ElemOf<C>::T;
  const SvdMat mt = mats[blockIdx.y];
  const T *a = static_cast<const T *>(a_) + mt.a_off;
  T *X = static_cast<T *>(ws_) + mt.x_off;
  T *V = static_cast<T *>(ws_) + mt.v_off;
  const int64_t MN = mt.M * mt.N, NN = mt.N * mt.N;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  for (int64_t e = blockIdx.x * kThreads + threadIdx.x; e < MN; e += stride) {
    const int64_t j = e / mt.M, i = e - j * mt.M;   // X(i, j) column-major
    X[e] = mt.tr ? conj_(a[e]) : a[i * mt.n + j];
  }
  for (int64_t e = blockIdx.x * kThreads + threadIdx.x; e < NN; e += stride) {
    const int64_t j = e / mt.N, i = e - j * mt.N;
    V[e] = (i == j) ? one_<T>() : zero_<T>();
  }
  for (int64_t e = blockIdx.x * kThreads + threadIdx.x; e < mt.N; e += stride)
    perm[mt.p_off + e] = static_cast<int32_t>(e);
}

// Squared column norms of the working matrices, one wave per column:
// grid (column groups of kWaves, matrices); `all` = 0 skips the matrices
// that have converged.  norms[p_off + c] = |X_c|^2.
template <bool C>
__global__ void __launch_bounds__(kThreads) k_svd_norms(const SvdMat *mats, const void *ws_, const int32_t *active,
                                                         int32_t all, double *norms) {
  using T = typename ElemOf<C>::T;
  const int mi = blockIdx.y;
  if (!all && !active[mi]) return;
  const SvdMat mt = mats[mi];
  const int64_t c = int64_t(blockIdx.x) * kWaves + (threadIdx.x >> 6);
  if (c >= mt.N) return;
  const int lane = threadIdx.x & 63;
  const T *col = static_cast<const T *>(ws_) + mt.x_off + c * mt.M;
  double acc = 0.0;
  for (int64_t i = lane; i < mt.M; i += 64) acc += abs2_(col[i]);
  acc = wave_sum(acc);
  if (lane == 0) norms[mt.p_off + c] = acc;
}

// The matrix's squared column norms into sn[0..N), then ord[rank] = column
// by decreasing norm (ties by column index; a NaN norm counts as the least, so
// that every rank is taken once and the order stays a permutation).
__device__ void order_by_norms(const double *norms, int64_t N, double *sn, int32_t *ord) {
  for (int64_t c = threadIdx.x; c < N; c += kThreads) sn[c] = norms[c] >= 0.0 ? norms[c] : -1.0;
  __syncthreads();
  for (int64_t c = threadIdx.x; c < N; c += kThreads) {
    const double v = sn[c];
    int32_t rank = 0;
    for (int64_t j = 0; j < N; ++j) {
      const double w = sn[j];
      rank += (w > v) || (w == v && j < c);
    }
    ord[rank] = static_cast<int32_t>(c);
  }
  __syncthreads();
}

// Column order of the next sweep: the physical columns by decreasing norm
// (the new order is a permutation of physical columns, so the previous order
// is not read).
__global__ void __launch_bounds__(kThreads) k_svd_sort(const SvdMat *mats, const double *norms, int32_t *perm,
                                                        const int32_t *active, int32_t all) {
  __shared__ double sn[kMaxSortCols];
  __shared__ int32_t so[kMaxSortCols];
  const int mi = blockIdx.x;
  if (!all && !active[mi]) return;
  const SvdMat mt = mats[mi];
  if (mt.N > kMaxSortCols) return;   // keep the previous order
  order_by_norms(norms + mt.p_off, mt.N, sn, so);
  for (int64_t c = threadIdx.x; c < mt.N; c += kThreads) perm[mt.p_off + c] = so[c];
}

// The pair (bi, bj) of round `round`, its column count w and its columns.
// Returns false when the matrix sits this round out or the pair has < 2 columns.
__device__ __forceinline__ bool pair_cols(const SvdMat &mt, int32_t round, int32_t k, const int32_t *perm,
                                          int32_t *sCol, int &w) {
  if (round >= mt.P - 1) return false;
  int bi, bj;
  circle_pair(mt.P, round, k, bi, bj);
  const int wi = bi < mt.nb ? static_cast<int>(min<int64_t>(kB, mt.N - int64_t(bi) * kB)) : 0;
  const int wj = bj < mt.nb ? static_cast<int>(min<int64_t>(kB, mt.N - int64_t(bj) * kB)) : 0;
  w = wi + wj;
  if (w < 2) return false;
  const int32_t *pm = perm + mt.p_off;
  const int tid = threadIdx.x;
  if (tid < w) sCol[tid] = tid < wi ? pm[int64_t(bi) * kB + tid] : pm[int64_t(bj) * kB + (tid - wi)];
  return true;
}

// Stage rows rb .. re of the panel's w columns (column c = X column sCol[c])
// into LDS as real and imaginary planes sP[part][c][row], zero beyond the
// rows and columns.  The loads carry no guards (past the panel they read its
// last row or column): guarded, each was waited for before the next (a Gram
// launch of the D = 2048 complex128 SVD 10.8 -> 9.7 us).
template <bool C, int R, int NT, typename T>
__device__ __forceinline__ void stage_panel(const T *base, int64_t rows, int64_t rb, int64_t re, int w,
                                            const int32_t *sCol, double (*sP)[kW][R + 1]) {
  constexpr int kCols = NT / R;   // columns per pass: consecutive threads take consecutive rows
  const int rr = threadIdx.x % R, c0 = threadIdx.x / R;
  const int64_t row = min<int64_t>(rb + rr, re - 1);
  T v[kW / kCols];
#pragma unroll
  for (int j = 0; j < kW / kCols; ++j) v[j] = base[int64_t(sCol[min(c0 + j * kCols, w - 1)]) * rows + row];
#pragma unroll
  for (int j = 0; j < kW / kCols; ++j) {
    const int c = c0 + j * kCols;
    const bool in = c < w && rb + rr < re;
    if constexpr (C) {
      sP[0][c][rr] = in ? v[j].x : 0.0;
      sP[1][c][rr] = in ? v[j].y : 0.0;
    } else {
      sP[0][c][rr] = in ? v[j] : 0.0;
    }
  }
}

// Round phase 1: one row group's part of the pair's Gram matrix, G = P^H P over rows
// g kRG .. (g + 1) kRG - 1, on v_mfma_f64_16x16x4f64: wave wv computes the
// 16 x 16 tile (wv / 2, wv % 2) of the 32 x 32 result over 16 k-steps of 4
// rows.  Complex: Re G = Pr^T Pr + Pi^T Pi, Im G = Pr^T Pi - Pi^T Pr.
template <bool C, int NT>
__device__ __forceinline__ void gram_tile(const SvdMat &mt, int32_t g, const void *ws_, int w, const int32_t *sCol,
                                          double (*sP)[kW][kRG + 1], v4d &acc, v4d &acc_i) {
  using T = typename ElemOf<C>::T;
  const int tid = threadIdx.x;
  const T *X = static_cast<const T *>(ws_) + mt.x_off;
  const int64_t rb = int64_t(g) * kRG, re = min<int64_t>(mt.M, rb + kRG);
  stage_panel<C, kRG, NT>(X, mt.M, rb, re, w, sCol, sP);
  __syncthreads();
  const int lane = tid & 63, wv = tid >> 6, lr = lane & 15, lk = lane >> 4;
  const int p0 = 16 * (wv >> 1), q0 = 16 * (wv & 1);
  acc = acc_i = v4d{0.0, 0.0, 0.0, 0.0};
  if (p0 >= w || q0 >= w) return;   // waves past the four tiles have p0 >= kW
#pragma unroll 4
  for (int ks = 0; ks < kRG; ks += 4) {
    const double ar = sP[0][p0 + lr][ks + lk], br = sP[0][q0 + lr][ks + lk];
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, acc, 0, 0, 0);
    if constexpr (C) {
      const double ai = sP[1][p0 + lr][ks + lk], bi = sP[1][q0 + lr][ks + lk];
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, bi, acc, 0, 0, 0);
      acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, acc_i, 0, 0, 0);
      acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, br, acc_i, 0, 0, 0);
    }
  }
}

// The thread's 4 entries of its wave's tile, put(p, q, value).
template <bool C, typename F>
__device__ __forceinline__ void each_gram_entry(int w, const v4d &acc, const v4d &acc_i, F put) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int p = 16 * (wv >> 1) + 4 * v + lk, q = 16 * (wv & 1) + lr;
    if (p < w && q < w) {
      if constexpr (C) put(p, q, cplx{acc[v], acc_i[v]});
      else put(p, q, acc[v]);
    }
  }
}

template <bool C>
__global__ void __launch_bounds__(kThreads) k_svd_gram(const SvdMat *mats, const SvdRowItem *items, int32_t round,
                                                        const void *ws_, const int32_t *perm, const int32_t *active,
                                                        void *part_) {
  using T = typename ElemOf<C>::T;
  __shared__ double sP[C ? 2 : 1][kW][kRG + 1];
  __shared__ int32_t sCol[kW];
  const SvdRowItem it = items[blockIdx.x];
  const SvdMat mt = mats[it.mat];
  if (!active[it.mat]) return;
  int w = 0;
  if (!pair_cols(mt, round, it.k, perm, sCol, w)) return;
  __syncthreads();
  v4d acc, acc_i;
  gram_tile<C, kThreads>(mt, it.g, ws_, w, sCol, sP, acc, acc_i);
  T *part = static_cast<T *>(part_) + (mt.gram0 + int64_t(it.k) * mt.ng + it.g) * (kW * kW);
  each_gram_entry<C>(w, acc, acc_i, [&](int p, int q, T v) { part[p * kW + q] = v; });
}

// Round phase 2, one workgroup per pair: the Gram matrix as the sum of the
// row groups' partials (in group order), the pair's convergence test, and one
// sweep of the cyclic two-sided Jacobi eigen-solve of the Gram in LDS, whose
// unitary Q (w x w, row stride kW) phase 3 applies.  qflag = 1 when Q is to be
// applied.
//
// What bounds it: the chain of each of the sweep's w - 1 rounds (read G, a
// rotation's square roots and divisions, apply, write G, barrier), with one
// workgroup per pair and far fewer pairs than CUs.  So everything that is
// not on that chain is kept off it: Q has waves of its own, which share the
// SIMDs with the chain's; a thread's column rotation is the one its lane has
// computed, only the row rotation comes by shuffle; the entries of G a thread
// works on are read before the rotation is known.
// GRAM: the workgroup forms the pair's Gram itself, phase 1 and 2 in one
// launch, for calls whose matrices have one row group each (a 33 x 32 matrix,
// complex128: 853 -> 653 us, FP64 706 -> 595); with more groups the last
// workgroup of a pair to write its part would have to go on, and the
// device-wide fences of all of them took 72 us a round in the D = 2048 SVD where
// the two launches take 39.
// A visit in a U(1)xU(1) D = 2048
// complex128 SVD: 47.6 us with G and Q in the same waves and all rotations by
// shuffle, 37.2 with waves for Q, 29.6 with the rows of kS entries; of a round's
// 1.0 us a rotation's square roots and divisions are 0.4.
// Row stride of G and Q in LDS: even, so that the entries (p, q) and (p, p) of
// the 16 pairs of a round, which lie along an antidiagonal and the diagonal,
// fall into different banks.
constexpr int kS = kW + 2;

// A sweep applies, round by round, the rotations of P2 / 2 disjoint index
// pairs, G <- J^H G J and Q <- Q J, as 2 x 2 blocks: thread (bi, bj) of the
// waves of G takes the block of G at rows (p, q) of pair bi and columns of
// pair bj, applies the rotation of pair bj to its columns and then that of
// pair bi to its rows (the same operations, in the same order, as a column
// pass followed by a row pass), and writes the result into the other G
// buffer; thread (bi, bj) of the waves of Q rotates rows 2 bi, 2 bi + 1 of Q
// in the columns of pair bj, in place.  Every wave computes the round's
// rotations from the round's G, pair k in lane k (and its copies k + 16, ...),
// so that a lane's own is that of pair bj, and a round takes one barrier: both
// kinds of waves pass the same number of them.  w odd: the pair with index w
// is off, and what stands in its row and column of G reaches no other.
template <bool C, bool FORQ, typename T = typename ElemOf<C>::T>
__device__ __forceinline__ void jacobi_sweep(T (*sG)[kW][kS], T (*sQ)[kS], int w) {
  const int P2 = w + (w & 1);
  const double eps = 2.220446049250313e-16;
  const int bi = (threadIdx.x % (kSolveThreads / 2)) / (kW / 2), bj = threadIdx.x % (kW / 2);
  const bool blk_on = bi < P2 / 2 && bj < P2 / 2;
  const int ki = min(bi, P2 / 2 - 1), kj = min(bj, P2 / 2 - 1);   // in range: nothing of other threads is stored
  int cur = 0;
  for (int r = 0; r < P2 - 1; ++r) {
    const T(*G)[kS] = sG[cur];
    int rows[2], cols[2];
    circle_pair(P2, r, kj, cols[0], cols[1]);
    if (FORQ) {
      rows[0] = 2 * ki;
      rows[1] = 2 * ki + 1;
    } else {
      circle_pair(P2, r, ki, rows[0], rows[1]);
    }
    const double al = re_(G[cols[0]][cols[0]]), be = re_(G[cols[1]][cols[1]]);
    const T g = G[cols[0]][cols[1]];
    T x[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) x[a][b] = FORQ ? sQ[rows[a]][cols[b]] : G[rows[a]][cols[b]];
    // the rotation of pair bj: c, s and the unit phase; off (identity) when
    // the pair is orthogonal or padded.  |g| > eps sqrt(al be), squared: three
    // square roots and three divisions per rotation.
    const double ag2 = sq_(g);
    const bool onj = (cols[0] < w) & (cols[1] < w) & (ag2 > 0.0) & (al > 0.0) & (be > 0.0) &
                     (ag2 > (eps * eps) * (al * be));
    const double ag = sqrt(ag2);
    const double inv = 1.0 / ag;
    const double zeta = (be - al) * (0.5 * inv);
    const bool far = fabs(zeta) > 1e150;
    const double num = far ? 0.5 : (zeta >= 0.0 ? 1.0 : -1.0);
    const double den = far ? zeta : fabs(zeta) + sqrt(fma(zeta, zeta, 1.0));
    const double t = num / den;
    const double cj = 1.0 / sqrt(fma(t, t, 1.0));
    const double sj = cj * t;
    const T emj = uphase_conj_inv(g, inv);
    double ci = 0.0, si = 0.0;
    T emi = emj;
    bool oni = false;
    if (!FORQ) {
      ci = __shfl(cj, bi);
      si = __shfl(sj, bi);
      emi = shfl_(emj, bi);
      oni = __shfl(onj ? 1 : 0, bi) != 0;
    }
    // columns:  [x_p, x_q] <- [x_p, x_q] J,  J = [[c, s], [-s e^{-i phi}, c e^{-i phi}]]
    if (onj) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const T xp = x[a][0], emxq = phase_(emj, x[a][1]);
        x[a][0] = rot_p(cj, sj, xp, emxq);
        x[a][1] = rot_q(cj, sj, xp, emxq);
      }
    }
    if (FORQ) {
      if (blk_on && onj) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          if (rows[a] >= w) continue;
          sQ[rows[a]][cols[0]] = x[a][0];
          sQ[rows[a]][cols[1]] = x[a][1];
        }
      }
    } else {
      // rows:  [g_p; g_q] <- J^H [g_p; g_q]; the pair's own off-diagonal entries become 0
      if (oni) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const T gp = x[0][b], epgq = cphase_(emi, x[1][b]);
          T np = rot_p(ci, si, gp, epgq);
          T nq = rot_q(ci, si, gp, epgq);
          if (cols[b] == rows[1]) np = zero_<T>();
          if (cols[b] == rows[0]) nq = zero_<T>();
          x[0][b] = np;
          x[1][b] = nq;
        }
      }
      if (blk_on) {
        T(*Gn)[kS] = sG[cur ^ 1];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b) Gn[rows[a]][cols[b]] = x[a][b];
      }
    }
    __syncthreads();
    cur ^= 1;
  }
}

template <bool C, bool GRAM>
__global__ void __launch_bounds__(kSolveThreads) k_svd_solve(const SvdMat *mats, const SvdItem *items, int32_t round,
                                                              const void *ws_, const void *part_, const int32_t *perm,
                                                              const int32_t *active, void *q_, int32_t *qflag,
                                                              int32_t *rotated) {
  using T = typename ElemOf<C>::T;
  constexpr int PARTS = C ? 2 : 1;
  // G (of the current round, and the next) and Q; before them the panel
  constexpr size_t kG = 2 * kW * kS * sizeof(T), kQ = kW * kS * sizeof(T);
  static_assert(PARTS * kW * (kRG + 1) * sizeof(double) <= kG + kQ, "the panel fits in the place of G and Q");
  __shared__ __align__(16) char smem[kG + kQ];
  __shared__ int32_t sCol[kW];
  __shared__ double sRed[kSolveThreads / 64];
  auto *sG = reinterpret_cast<T(*)[kW][kS]>(smem);
  auto *sQ = reinterpret_cast<T(*)[kS]>(smem + kG);
  static_assert(kW == 32 && kSolveThreads == 512, "one thread per 2 x 2 block of pairs, for G and for Q");
  constexpr int kPer = kW * kW / kSolveThreads;

  const SvdItem it = items[blockIdx.x];
  const SvdMat mt = mats[it.mat];
  if (!active[it.mat]) return;
  const int tid = threadIdx.x;
  int w = 0;
  if (!pair_cols(mt, round, it.k, perm, sCol, w)) return;
  int32_t *flag = qflag + mt.pair0 + it.k;
  if constexpr (GRAM) {
    __syncthreads();
    v4d acc, acc_i;
    gram_tile<C, kSolveThreads>(mt, 0, ws_, w, sCol, reinterpret_cast<double(*)[kW][kRG + 1]>(smem), acc, acc_i);
    __syncthreads();   // the panel is read: G and Q take its place
    each_gram_entry<C>(w, acc, acc_i, [&](int p, int q, T v) { sG[0][p][q] = add_(zero_<T>(), v); });
  } else {
    const T *part = static_cast<const T *>(part_) + (mt.gram0 + int64_t(it.k) * mt.ng) * (kW * kW);
    T sum[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) sum[u] = zero_<T>();
    for (int g = 0; g < mt.ng; ++g)   // entries past w x w: whatever the slot holds, not used
#pragma unroll
      for (int u = 0; u < kPer; ++u) sum[u] = add_(sum[u], part[int64_t(g) * (kW * kW) + tid + u * kSolveThreads]);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int e = tid + u * kSolveThreads;
      sG[0][e / kW][e % kW] = sum[u];
    }
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int e = tid + u * kSolveThreads, p = e / kW, q = e % kW;
    sQ[p][q] = (p == q) ? one_<T>() : zero_<T>();
  }
  __syncthreads();

  // ---- convergence test of the pair ----
  double off = 0.0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int e = tid + u * kSolveThreads, p = e / kW, q = e % kW;
    if (p < q && q < w) {
      const double dp = re_(sG[0][p][p]), dq = re_(sG[0][q][q]);
      if (dp > 0.0 && dq > 0.0) off = fmax(off, abs2_(sG[0][p][q]) / (dp * dq));
    }
  }
  off = wave_max(off);
  if ((tid & 63) == 0) sRed[tid >> 6] = off;
  __syncthreads();
  const double tol = fmax(16.0, static_cast<double>(mt.M)) * 2.220446049250313e-16;
  double offmax = sRed[0];
#pragma unroll
  for (int v = 1; v < kSolveThreads / 64; ++v) offmax = fmax(offmax, sRed[v]);
  if (offmax < tol * tol) {
    if (tid == 0) *flag = 0;
    return;
  }
  if (tid == 0) {
    rotated[it.mat] = 1;
    *flag = 1;
  }

  if (__builtin_amdgcn_readfirstlane(tid) < kSolveThreads / 2) jacobi_sweep<C, false>(sG, sQ, w);
  else jacobi_sweep<C, true>(sG, sQ, w);
  T *Q = static_cast<T *>(q_) + int64_t(mt.pair0 + it.k) * (kW * kW);
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int e = tid + u * kSolveThreads, p = e / kW, q = e % kW;
    if (p < w && q < w) Q[e] = sQ[p][q];
  }
}

// Round phase 3: P <- P Q for one group of kUR rows of the pair's columns of X
// (kind 0) or of V (kind 1), on v_mfma_f64_16x16x4f64 over k-steps of 4 of the
// pair's w columns: wave wv computes rows 16 (wv % 2) .. + 15 of columns
// 16 (wv / 2) .. + 15.  Complex: Re = Pr Qr - Pi Qi, Im = Pr Qi + Pi Qr.  The
// product is formed as Q^T P^T, whose accumulators hold consecutive rows in
// consecutive lanes, so that a store covers 256 bytes of each of 4 columns;
// as P Q, 64 bytes of each of 16, the stores took 6 of 16 us.  In a U(1)xU(1) D =
// 2048 complex128 SVD with guarded loads 17.7 us, unguarded 14.9, now 12.9; 4.5
// of it is a launch that finds nothing to do.
template <bool C>
__global__ void __launch_bounds__(kThreads) k_svd_update(const SvdMat *mats, const SvdRowItem *items, int32_t round,
                                                          void *ws_, const int32_t *perm, const int32_t *active,
                                                          const void *q_, const int32_t *qflag) {
  using T = typename ElemOf<C>::T;
  constexpr int PARTS = C ? 2 : 1;
  __shared__ double sP[PARTS][kW][kUR + 1];
  __shared__ double sQ[PARTS][kW][kW];
  __shared__ int32_t sCol[kW];
  const SvdRowItem it = items[blockIdx.x];
  const SvdMat mt = mats[it.mat];
  if (!active[it.mat]) return;
  int w = 0;
  if (!pair_cols(mt, round, it.k, perm, sCol, w)) return;
  if (!qflag[mt.pair0 + it.k]) return;
  const int tid = threadIdx.x;
  const T *Q = static_cast<const T *>(q_) + int64_t(mt.pair0 + it.k) * (kW * kW);
  T qv[kW * kW / kThreads];   // past w x w: whatever the slot holds, staged as zero
#pragma unroll
  for (int u = 0; u < kW * kW / kThreads; ++u) qv[u] = Q[tid + u * kThreads];
  T *base = static_cast<T *>(ws_) + (it.kind ? mt.v_off : mt.x_off);
  const int64_t rows = it.kind ? mt.N : mt.M;
  const int64_t rb = int64_t(it.g) * kUR, re = min<int64_t>(rows, rb + kUR);
  __syncthreads();
  stage_panel<C, kUR, kThreads>(base, rows, rb, re, w, sCol, sP);
#pragma unroll
  for (int u = 0; u < kW * kW / kThreads; ++u) {
    const int e = tid + u * kThreads, p = e / kW, q = e % kW;
    const bool in = p < w && q < w;
    if constexpr (C) {
      sQ[0][p][q] = in ? qv[u].x : 0.0;
      sQ[1][p][q] = in ? qv[u].y : 0.0;
    } else {
      sQ[0][p][q] = in ? qv[u] : 0.0;
    }
  }
  __syncthreads();
  const int lane = tid & 63, wv = tid >> 6, lr = lane & 15, lk = lane >> 4;
  typedef double v4d __attribute__((ext_vector_type(4)));
  static_assert(kUR == 32 && kW == 32 && kWaves == 4, "one 16 x 16 tile per wave");
  const int r0 = 16 * (wv & 1), j0 = 16 * (wv >> 1);
  v4d acc = {0.0, 0.0, 0.0, 0.0}, acc_i = {0.0, 0.0, 0.0, 0.0};
  if (rb + r0 >= re || j0 >= w) return;
  for (int ks = 0; ks < w; ks += 4) {
    const double ar = sP[0][ks + lk][r0 + lr], br = sQ[0][ks + lk][j0 + lr];
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(br, ar, acc, 0, 0, 0);
    if constexpr (C) {
      const double ai = sP[1][ks + lk][r0 + lr], bi = sQ[1][ks + lk][j0 + lr];
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(bi, -ai, acc, 0, 0, 0);
      acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(bi, ar, acc_i, 0, 0, 0);
      acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(br, ai, acc_i, 0, 0, 0);
    }
  }
  // every read of the rows is done (they sit in LDS): write the new columns
  const int64_t row = rb + r0 + lr;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int j = j0 + 4 * v + lk;
    if (row < re && j < w) {
      T *dst = base + int64_t(sCol[j]) * rows + row;
      if constexpr (C) *dst = cplx{acc[v], acc_i[v]};
      else *dst = acc[v];
    }
  }
}

// Singular values and vectors, grid (element groups, matrices): the columns
// in the order of `ord` (decreasing norm, written by k_svd_sort), sigma_k =
// sqrt(norm of column ord[k]).
template <bool C>
__global__ void __launch_bounds__(kThreads) k_svd_finish(const SvdMat *mats, const void *ws_, const double *norms,
                                                          const int32_t *ord, void *u_, double *s_, void *vt_) {
  using T = typename ElemOf<C>::T;
  const SvdMat mt = mats[blockIdx.y];
  const T *X = static_cast<const T *>(ws_) + mt.x_off;
  const T *V = static_cast<const T *>(ws_) + mt.v_off;
  const double *nm = norms + mt.p_off;
  const int32_t *so = ord + mt.p_off;
  T *U = static_cast<T *>(u_) + mt.u_off;
  T *Vt = static_cast<T *>(vt_) + mt.vt_off;
  double *S = s_ + mt.s_off;
  const int64_t r = mt.N;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  const int64_t e0 = blockIdx.x * kThreads + threadIdx.x;
  for (int64_t k = e0; k < r; k += stride) S[k] = sqrt(nm[so[k]]);
  if (!mt.tr) {
    // A = X_final V^H:  U (m x r) = X_col / sigma, Vt (r x n) = V^H
    for (int64_t e = e0; e < mt.m * r; e += stride) {
      const int64_t i = e / r, k = e - i * r;
      const int32_t c = so[k];
      const double sg = sqrt(nm[c]);
      U[e] = sg > 0.0 ? scl_(1.0 / sg, X[int64_t(c) * mt.M + i]) : zero_<T>();
    }
    for (int64_t e = e0; e < r * mt.n; e += stride) {
      const int64_t k = e / mt.n, j = e - k * mt.n;
      Vt[e] = conj_(V[int64_t(so[k]) * mt.N + j]);
    }
  } else {
    // A^H = X_final V^H  =>  A = V X_final^H:  U (m x r) = V, Vt (r x n) = (X_col / sigma)^H
    for (int64_t e = e0; e < mt.m * r; e += stride) {
      const int64_t i = e / r, k = e - i * r;
      U[e] = V[int64_t(so[k]) * mt.N + i];
    }
    for (int64_t e = e0; e < r * mt.n; e += stride) {
      const int64_t k = e / mt.n, j = e - k * mt.n;
      const int32_t c = so[k];
      const double sg = sqrt(nm[c]);
      Vt[e] = sg > 0.0 ? scl_(1.0 / sg, conj_(X[int64_t(c) * mt.M + j])) : zero_<T>();
    }
  }
}

template <bool C>
qlt_status svd_impl(int64_t n_mats, const int64_t *rows, const int64_t *cols, const void *a, const int64_t *a_offsets,
                    void *u, const int64_t *u_offsets, double *s, const int64_t *s_offsets, void *vt,
                    const int64_t *vt_offsets, int32_t *sweeps_out, hipStream_t st) {
  const size_t esz = C ? 16 : 8;
  QLT_CHECK_ARG(n_mats <= 65535, "qlt_block_svd: more than 65535 matrices in one call");
  std::vector<SvdMat> mats(static_cast<size_t>(n_mats));
  std::vector<SvdItem> items;
  std::vector<SvdRowItem> gitems, uitems;
  int64_t ws_elems = 0, perm_elems = 0, max_elems = 0, gram_slots = 0;
  int32_t max_players = 0, pair_slots = 0;
  for (int64_t i = 0; i < n_mats; ++i) {
    SvdMat &mt = mats[static_cast<size_t>(i)];
    mt.m = rows[i];
    mt.n = cols[i];
    mt.tr = rows[i] < cols[i];
    mt.M = std::max(rows[i], cols[i]);
    mt.N = std::min(rows[i], cols[i]);
    QLT_CHECK_ARG(mt.N <= kMaxSortCols, "qlt_block_svd: min(rows, cols) of matrix " + std::to_string(i) +
                                            " exceeds " + std::to_string(kMaxSortCols));
    mt.x_off = ws_elems;
    ws_elems += mt.M * mt.N;
    mt.v_off = ws_elems;
    ws_elems += mt.N * mt.N;
    mt.p_off = perm_elems;
    perm_elems += mt.N;
    mt.a_off = a_offsets[i];
    mt.u_off = u_offsets[i];
    mt.s_off = s_offsets[i];
    mt.vt_off = vt_offsets[i];
    mt.nb = static_cast<int32_t>((mt.N + kB - 1) / kB);
    mt.P = mt.nb == 1 ? 2 : mt.nb + (mt.nb & 1);
    mt.ng = static_cast<int32_t>((mt.M + kRG - 1) / kRG);
    mt.pair0 = pair_slots;
    mt.pad = 0;
    mt.gram0 = gram_slots;
    max_elems = std::max(max_elems, mt.M * mt.N);
    if (mt.N >= 2) {
      max_players = std::max(max_players, mt.P);
      const int32_t nux = static_cast<int32_t>((mt.M + kUR - 1) / kUR), nuv = static_cast<int32_t>((mt.N + kUR - 1) / kUR);
      for (int32_t k = 0; k < mt.P / 2; ++k) {
        items.push_back(SvdItem{static_cast<int32_t>(i), k});
        for (int32_t g = 0; g < mt.ng; ++g) gitems.push_back(SvdRowItem{static_cast<int32_t>(i), k, g, 0});
        for (int32_t g = 0; g < nux; ++g) uitems.push_back(SvdRowItem{static_cast<int32_t>(i), k, g, 0});
        for (int32_t g = 0; g < nuv; ++g) uitems.push_back(SvdRowItem{static_cast<int32_t>(i), k, g, 1});
      }
      pair_slots += mt.P / 2;
      gram_slots += int64_t(mt.P / 2) * mt.ng;
    }
  }
  QLT_CHECK_ARG(gitems.size() < (size_t(1) << 31) && uitems.size() < (size_t(1) << 31),
                "qlt_block_svd: too many row groups in one call");
  DevBuf d_ws, d_mats, d_items, d_perm, d_flags, d_gitems, d_uitems, d_part, d_q, d_qflag, d_norms;
  QLT_HIP(hipMalloc(&d_ws.p, std::max<size_t>(1, static_cast<size_t>(ws_elems) * esz)));
  QLT_HIP(hipMalloc(&d_mats.p, sizeof(SvdMat) * mats.size()));
  QLT_HIP(hipMalloc(&d_items.p, sizeof(SvdItem) * std::max<size_t>(1, items.size())));
  QLT_HIP(hipMalloc(&d_gitems.p, sizeof(SvdRowItem) * std::max<size_t>(1, gitems.size())));
  QLT_HIP(hipMalloc(&d_uitems.p, sizeof(SvdRowItem) * std::max<size_t>(1, uitems.size())));
  QLT_HIP(hipMalloc(&d_part.p, esz * kW * kW * static_cast<size_t>(std::max<int64_t>(1, gram_slots))));
  QLT_HIP(hipMalloc(&d_q.p, esz * kW * kW * static_cast<size_t>(std::max<int32_t>(1, pair_slots))));
  QLT_HIP(hipMalloc(&d_qflag.p, sizeof(int32_t) * static_cast<size_t>(std::max<int32_t>(1, pair_slots))));
  QLT_HIP(hipMalloc(&d_perm.p, sizeof(int32_t) * std::max<int64_t>(1, perm_elems)));
  QLT_HIP(hipMalloc(&d_norms.p, sizeof(double) * std::max<int64_t>(1, perm_elems)));
  QLT_HIP(hipMalloc(&d_flags.p, sizeof(int32_t) * 2 * mats.size()));
  auto *active = static_cast<int32_t *>(d_flags.p);
  auto *rotated = active + mats.size();
  QLT_HIP(hipMemcpyAsync(d_mats.p, mats.data(), sizeof(SvdMat) * mats.size(), hipMemcpyHostToDevice, st));
  if (!items.empty()) {
    QLT_HIP(hipMemcpyAsync(d_items.p, items.data(), sizeof(SvdItem) * items.size(), hipMemcpyHostToDevice, st));
    QLT_HIP(hipMemcpyAsync(d_gitems.p, gitems.data(), sizeof(SvdRowItem) * gitems.size(), hipMemcpyHostToDevice,
                           st));
    QLT_HIP(hipMemcpyAsync(d_uitems.p, uitems.data(), sizeof(SvdRowItem) * uitems.size(), hipMemcpyHostToDevice,
                           st));
  }
  const auto *gi = static_cast<const SvdRowItem *>(d_gitems.p);
  const auto *ui = static_cast<const SvdRowItem *>(d_uitems.p);
  auto *qflag = static_cast<int32_t *>(d_qflag.p);
  const auto *dm = static_cast<const SvdMat *>(d_mats.p);
  auto *perm = static_cast<int32_t *>(d_perm.p);
  auto *norms = static_cast<double *>(d_norms.p);
  int64_t max_n = 1;
  for (const SvdMat &mt : mats) max_n = std::max(max_n, mt.N);
  const dim3 norms_grid(static_cast<unsigned>((max_n + kWaves - 1) / kWaves), static_cast<unsigned>(n_mats));
  const unsigned gx = static_cast<unsigned>(std::min<int64_t>(1024, std::max<int64_t>(1, (max_elems + kThreads - 1) / kThreads)));
  hipLaunchKernelGGL(k_svd_load<C>, dim3(gx, static_cast<unsigned>(n_mats)), dim3(kThreads), 0, st, dm, a,
                     d_ws.p, perm);
  QLT_HIP(hipGetLastError());
  std::vector<int32_t> h_active(mats.size()), h_rot(mats.size(), 0);
  for (size_t i = 0; i < mats.size(); ++i) h_active[i] = mats[i].N >= 2;
  int32_t sweeps = 0;
  bool any = !items.empty(), one_group = true;   // one row group per matrix of more than one column
  for (const SvdMat &mt : mats) one_group = one_group && (mt.N < 2 || mt.ng == 1);
  while (any && sweeps < kMaxSweeps) {
    QLT_HIP(hipMemcpyAsync(active, h_active.data(), sizeof(int32_t) * mats.size(), hipMemcpyHostToDevice, st));
    std::fill(h_rot.begin(), h_rot.end(), 0);
    QLT_HIP(hipMemcpyAsync(rotated, h_rot.data(), sizeof(int32_t) * mats.size(), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_svd_norms<C>, norms_grid, dim3(kThreads), 0, st, dm, d_ws.p, active, 0, norms);
    hipLaunchKernelGGL(k_svd_sort, dim3(static_cast<unsigned>(n_mats)), dim3(kThreads), 0, st, dm, norms, perm,
                       active, 0);
    for (int32_t r = 0; r < max_players - 1; ++r) {
      if (!one_group)
        hipLaunchKernelGGL(k_svd_gram<C>, dim3(static_cast<unsigned>(gitems.size())), dim3(kThreads), 0, st, dm, gi, r,
                           d_ws.p, perm, active, d_part.p);
      hipLaunchKernelGGL((one_group ? k_svd_solve<C, true> : k_svd_solve<C, false>),
                         dim3(static_cast<unsigned>(items.size())), dim3(kSolveThreads), 0, st, dm,
                         static_cast<const SvdItem *>(d_items.p), r, d_ws.p, d_part.p, perm, active, d_q.p, qflag,
                         rotated);
      hipLaunchKernelGGL(k_svd_update<C>, dim3(static_cast<unsigned>(uitems.size())), dim3(kThreads), 0, st, dm, ui,
                         r, d_ws.p, perm, active, d_q.p, qflag);
    }
    QLT_HIP(hipGetLastError());
    QLT_HIP(hipMemcpyAsync(h_rot.data(), rotated, sizeof(int32_t) * mats.size(), hipMemcpyDeviceToHost, st));
    QLT_HIP(hipStreamSynchronize(st));
    ++sweeps;
    any = false;
    for (size_t i = 0; i < mats.size(); ++i) {
      h_active[i] = h_active[i] && h_rot[i];
      any = any || h_active[i];
    }
  }
  // final order of every matrix (into the column-order buffer), then U, S, V^H
  hipLaunchKernelGGL(k_svd_norms<C>, norms_grid, dim3(kThreads), 0, st, dm, d_ws.p, active, 1, norms);
  hipLaunchKernelGGL(k_svd_sort, dim3(static_cast<unsigned>(n_mats)), dim3(kThreads), 0, st, dm, norms, perm, active,
                     1);
  hipLaunchKernelGGL(k_svd_finish<C>, dim3(gx, static_cast<unsigned>(n_mats)), dim3(kThreads), 0, st, dm, d_ws.p,
                     norms, perm, u, s, vt);
  QLT_HIP(hipGetLastError());
  QLT_HIP(hipStreamSynchronize(st));
  if (sweeps_out != nullptr) *sweeps_out = sweeps;
  if (any) return qlt::fail(QLT_ERR_NOT_CONVERGED, "qlt_block_svd: Jacobi sweeps did not converge in " +
                                                        std::to_string(kMaxSweeps) + " sweeps");
  return QLT_OK;
}

}  // namespace

extern "C" {

qlt_status qlt_block_svd(int32_t dtype, int64_t n_mats, const int64_t *rows, const int64_t *cols, const void *a,
                         const int64_t *a_offsets, void *u, const int64_t *u_offsets, double *s,
                         const int64_t *s_offsets, void *vt, const int64_t *vt_offsets, int32_t *sweeps,
                         void *stream) {
  QLT_REQUIRE_INIT();
  QLT_CHECK_ARG(qlt::valid_dtype(dtype), "qlt_block_svd: bad dtype");
  QLT_TRY(check_shapes("qlt_block_svd", n_mats, rows, cols));
  if (sweeps != nullptr) *sweeps = 0;
  if (n_mats == 0) return QLT_OK;
  QLT_CHECK_ARG(a != nullptr && u != nullptr && s != nullptr && vt != nullptr, "qlt_block_svd: null data pointer");
  QLT_CHECK_ARG(a_offsets != nullptr && u_offsets != nullptr && s_offsets != nullptr && vt_offsets != nullptr,
                "qlt_block_svd: null offset array");
  QLT_CHECK_ARG(!qlt::stream_capturing(qlt::as_stream(stream)), "qlt_block_svd: not capturable (host-driven sweeps)");
  if (qlt::dtype_is_single(dtype)) {
    const int32_t wide = dtype == QLT_F32 ? QLT_F64 : QLT_C128;
    const int64_t esz = qlt::dtype_bytes(wide);
    std::vector<int64_t> kk(static_cast<size_t>(n_mats));
    for (int64_t i = 0; i < n_mats; ++i) kk[i] = std::min(rows[i], cols[i]);
    const int64_t na = extent(n_mats, a_offsets, rows, cols);
    const int64_t nu = extent(n_mats, u_offsets, rows, kk.data());
    const int64_t nv = extent(n_mats, vt_offsets, kk.data(), cols);
    DevBuf wa, wu, wv;
    QLT_HIP(hipMalloc(&wa.p, std::max<int64_t>(1, na) * esz));
    QLT_HIP(hipMalloc(&wu.p, std::max<int64_t>(1, nu) * esz));
    QLT_HIP(hipMalloc(&wv.p, std::max<int64_t>(1, nv) * esz));
    QLT_TRY(qlt_convert(dtype, wide, na, a, wa.p, stream));
    QLT_TRY(qlt_block_svd(wide, n_mats, rows, cols, wa.p, a_offsets, wu.p, u_offsets, s, s_offsets, wv.p,
                          vt_offsets, sweeps, stream));
    QLT_TRY(qlt_convert(wide, dtype, nu, wu.p, u, stream));
    QLT_TRY(qlt_convert(wide, dtype, nv, wv.p, vt, stream));
    QLT_HIP(hipStreamSynchronize(qlt::as_stream(stream)));
    return QLT_OK;
  }
  if (dtype == QLT_F64)
    return svd_impl<false>(n_mats, rows, cols, a, a_offsets, u, u_offsets, s, s_offsets, vt, vt_offsets, sweeps,
                           qlt::as_stream(stream));
  return svd_impl<true>(n_mats, rows, cols, a, a_offsets, u, u_offsets, s, s_offsets, vt, vt_offsets, sweeps,
                        qlt::as_stream(stream));
}

}  // extern "C"
