// Batched QR of the block matrices of a block-sparse tensor, in FP64 and
// complex128, by blocked Householder reflections.  It replaces MatQR
// (framework/hp_numeric/lapack.h:332-487 geqrf + orgqr / ungqr) called once per
// block matrix by DataBlkDecompQR (qltensor/blk_spar_data_ten/
// data_blk_operations.h:1028-1046); here every block matrix of the tensor is
// decomposed in one batched launch sequence.
//
// Reflectors follow LAPACK's convention (xLARFG: beta = -sign(Re alpha) *
// |(alpha, x)|, tau = (beta - alpha) / beta, v = x / (alpha - beta); no
// reflection when x = 0 and alpha is real), so R has the same diagonal signs
// as geqrf, and Q = H_0 ... H_{k-1} I[:, :k] as orgqr / ungqr form it.
//
// The columns are taken in blocks of kNB.  Launch b (k_qr_step) applies the
// reflectors of block b, I - V T V^H, to every later column tile, one
// workgroup per tile and matrix, and the workgroup that holds the next block
// goes on to factor it, so one launch per block is both the trailing update
// and the next panel.  A last launch (k_qr_q) writes R and applies the blocks
// to the identity, each Q tile on its own.  Both contractions of an
// application, V^H X and V (T V^H X), run on v_mfma_f64_16x16x4f64; a panel
// sits in registers, and one reduction per column gives at once the column's
// norm, its products with the later columns (the update) and with the earlier
// ones (the column of T).
//
// What bounds it: the chain of columns (one workgroup reduction and a square
// root and two divisions each, about 1.3 us) and of launches.  The unblocked
// form (k_qr_generic: one workgroup per matrix, every reflector a pass over
// the whole trailing matrix) reads the matrix k times through one compute
// unit: 17 FP64 matrices of up to 266 x 266 took 22.0 ms that way and take
// 0.66 ms in blocks (16 trailing launches of 28 us, 83 us for Q).

#include <algorithm>
#include <vector>

#include "block_dense.h"

using namespace qlt::dense;

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kNB = 16;   // columns per block: one MFMA tile

struct QrMat {
  int64_t m, n, k;
  int64_t w_off;      // W: m x n, row-major (column-major in k_qr_generic)
  int64_t v_off;      // block b's reflectors at v_off + b m kNB: m x v_cols row-major, rows from b kNB on
                      // (k_qr_generic: Q, column-major m x k)
  int64_t t_off;      // block b's T at t_off + b kNB kNB (k_qr_generic: tau)
  int64_t a_off, q_off, r_off;
};

// Reflectors of block b of a matrix with k of them.
__device__ __forceinline__ int block_cols(int64_t k, int64_t b) {
  return static_cast<int>(k - b * kNB < kNB ? k - b * kNB : kNB);
}

// Row stride of block b's reflectors: with PAD the last block, too, takes kNB
// columns (zeros past k), and the stride is a constant.  Padding is faster (U(1)
// D = 1024, FP64: 656 us, 672 without) and costs a matrix of few columns a multiple
// of its size in scratch, so qr_impl takes it where that is little.
template <bool PAD>
__device__ __forceinline__ int v_cols(int64_t k, int64_t b) {
  return PAD ? kNB : block_cols(k, b);
}

// X <- (I - V op(T) V^H) X for rows r0 .. m - 1 and `nc` columns of X, op(T) =
// T^H (`CONJT`, applying the adjoint) or T.  V (row stride ldv) and T are block-reflector
// storage (QrMat), X is row-major with leading dimension ld.
//   P = V^H X: the rows are the contracted extent; wave w takes k-steps w,
//   w + W, ... of 4 rows and the waves' partial 16 x 16 sums meet in LDS;
//   Z = op(T) P, one element per thread;
//   X -= V Z: wave w takes row blocks w, w + W, ...
template <bool C, int NW, bool CONJT, bool PAD, typename T>
__device__ void apply_block(const T *__restrict__ V, int ldv, const T *__restrict__ Tm, T *X, int64_t ld, int64_t r0,
                            int64_t m, int nc, T (*sPart)[kNB][kNB + 1], T (*sZ)[kNB + 1], T (*sT)[kNB + 1]) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lk = lane >> 4;
  const int64_t mm = m - r0;
  const int steps = static_cast<int>((mm + 3) / 4);
  for (int e = tid; e < kNB * kNB; e += 64 * NW) sT[e / kNB][e % kNB] = Tm[e];
  v4d acc = {0.0, 0.0, 0.0, 0.0}, acc_i = {0.0, 0.0, 0.0, 0.0};
  constexpr int U = 4;   // k-steps whose loads are in flight together
  for (int s0 = w; s0 < steps; s0 += NW * U) {
    T va[U], xa[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = r0 + 4 * int64_t(s0 + NW * u) + lk;
      const bool ok = r < m;
      va[u] = (ok && (PAD || lr < ldv)) ? V[r * ldv + lr] : zero_<T>();
      xa[u] = (ok && lr < nc) ? X[r * ld + lr] : zero_<T>();
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (C) {
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u].x, xa[u].x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u].y, xa[u].y, acc, 0, 0, 0);
        acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u].x, xa[u].y, acc_i, 0, 0, 0);
        acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(-va[u].y, xa[u].x, acc_i, 0, 0, 0);
      } else {
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u], xa[u], acc, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    if constexpr (C) sPart[w][4 * v + lk][lr] = cplx{acc[v], acc_i[v]};
    else sPart[w][4 * v + lk][lr] = acc[v];
  }
  __syncthreads();
  for (int e = tid; e < kNB * kNB; e += 64 * NW) {
    const int p = e / kNB, q = e % kNB;
    T s = sPart[0][p][q];
#pragma unroll
    for (int g = 1; g < NW; ++g) s = add_(s, sPart[g][p][q]);
    sZ[p][q] = s;
  }
  __syncthreads();
  // T is upper triangular, stored with its zeros
  T (*sY)[kNB + 1] = sPart[0];
  for (int e = tid; e < kNB * kNB; e += 64 * NW) {
    const int p = e / kNB, q = e % kNB;
    T s = zero_<T>();
#pragma unroll
    for (int l = 0; l < kNB; ++l) s = add_(s, CONJT ? cmul_(sT[l][p], sZ[l][q]) : mul_(sT[p][l], sZ[l][q]));
    sY[p][q] = s;
  }
  __syncthreads();
  T y[kNB / 4];
#pragma unroll
  for (int s = 0; s < kNB / 4; ++s) y[s] = sY[4 * s + lk][lr];
  const int rblocks = static_cast<int>((mm + 15) / 16);
  for (int rb = w; rb < rblocks; rb += NW) {
    const int64_t rv = r0 + 16 * int64_t(rb) + lr;
    T va[kNB / 4], old[4];
#pragma unroll
    for (int s = 0; s < kNB / 4; ++s)
      va[s] = (rv < m && (PAD || 4 * s + lk < ldv)) ? V[rv * ldv + 4 * s + lk] : zero_<T>();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t r = r0 + 16 * int64_t(rb) + 4 * v + lk;
      old[v] = (r < m && lr < nc) ? X[r * ld + lr] : zero_<T>();
    }
    v4d d = {0.0, 0.0, 0.0, 0.0}, d_i = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < kNB / 4; ++s) {
      if constexpr (C) {
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(va[s].x, y[s].x, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(-va[s].y, y[s].y, d, 0, 0, 0);
        d_i = __builtin_amdgcn_mfma_f64_16x16x4f64(va[s].x, y[s].y, d_i, 0, 0, 0);
        d_i = __builtin_amdgcn_mfma_f64_16x16x4f64(va[s].y, y[s].x, d_i, 0, 0, 0);
      } else {
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(va[s], y[s], d, 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t r = r0 + 16 * int64_t(rb) + 4 * v + lk;
      if (r < m && lr < nc) {
        if constexpr (C) X[r * ld + lr] = cplx{old[v].x - d[v], old[v].y - d_i[v]};
        else X[r * ld + lr] = old[v] - d[v];
      }
    }
  }
}

// Sums over the wave of 16 values per lane: lane l returns the sum of value
// l / 4.  Each stage halves the values a lane keeps: lanes l and its partner
// (l ^ 32, l ^ 16, then l ^ 8 and 7 - l within rows of 16 and 8) swap halves
// and add; the four lanes of a quad finish.
__device__ __forceinline__ double swap_add(double a, double b, bool by32) {
  const uint64_t ua = __double_as_longlong(a), ub = __double_as_longlong(b);
  uint32_t al = static_cast<uint32_t>(ua), ah = static_cast<uint32_t>(ua >> 32);
  uint32_t bl = static_cast<uint32_t>(ub), bh = static_cast<uint32_t>(ub >> 32);
  if (by32) {
    const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    al = l[0];
    bl = l[1];
    ah = h[0];
    bh = h[1];
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    al = l[0];
    bl = l[1];
    ah = h[0];
    bh = h[1];
  }
  return __longlong_as_double(static_cast<int64_t>((uint64_t(ah) << 32) | al)) +
         __longlong_as_double(static_cast<int64_t>((uint64_t(bh) << 32) | bl));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const uint64_t u = __double_as_longlong(v);
  const uint32_t l = __builtin_amdgcn_mov_dpp(static_cast<int>(u), CTRL, 0xf, 0xf, true);
  const uint32_t h = __builtin_amdgcn_mov_dpp(static_cast<int>(u >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(static_cast<int64_t>((uint64_t(h) << 32) | l));
}
constexpr int kDppRor8 = 0x128, kDppHalfMirror = 0x141, kDppXor1 = 0xB1, kDppXor2 = 0x4E;
__device__ __forceinline__ double wave_sums16(const double (&d)[kNB], int lane) {
  double a[8], b[4], c[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = swap_add(d[i], d[i + 8], true);     // value i + 8 (lane >= 32)
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = swap_add(a[i], a[i + 4], false);    // + 4 (lane & 16)
  const bool up8 = (lane & 8) != 0, up4 = (lane & 4) != 0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const double keep = up8 ? b[i + 2] : b[i], send = up8 ? b[i] : b[i + 2];
    c[i] = keep + dpp_move<kDppRor8>(send);
  }
  double v = (up4 ? c[1] : c[0]) + dpp_move<kDppHalfMirror>(up4 ? c[0] : c[1]);
  v += dpp_move<kDppXor1>(v);
  v += dpp_move<kDppXor2>(v);
  return v;
}
__device__ __forceinline__ cplx wave_sums16(const cplx (&d)[kNB], int lane) {
  double x[kNB], y[kNB];
#pragma unroll
  for (int i = 0; i < kNB; ++i) {
    x[i] = d[i].x;
    y[i] = d[i].y;
  }
  return {wave_sums16(x, lane), wave_sums16(y, lane)};
}
__device__ __forceinline__ double lane_value(double v, int src) {
  const uint64_t u = __double_as_longlong(v);
  const uint32_t l = __builtin_amdgcn_readlane(static_cast<int>(u), src);
  const uint32_t h = __builtin_amdgcn_readlane(static_cast<int>(u >> 32), src);
  return __longlong_as_double(static_cast<int64_t>((uint64_t(h) << 32) | l));
}
__device__ __forceinline__ cplx lane_value(cplx v, int src) { return {lane_value(v.x, src), lane_value(v.y, src)}; }

__device__ __forceinline__ double sel_(bool c, double a, double b) { return c ? a : b; }
__device__ __forceinline__ cplx sel_(bool c, cplx a, cplx b) { return {c ? a.x : b.x, c ? a.y : b.y}; }
// Orders one wave's LDS writes before its lanes' reads of each other's data.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Launch b of the factorisation, grid (matrices, column tiles b + 1 ..).
// FIRST (b = -1): the tiles are copied from the input into W, and tile 0 is
// factored.  Rows up to 64 NW RPT.
template <bool C, int NW, int RPT, bool FIRST, bool PAD>
__global__ void __launch_bounds__(64 * NW) k_qr_step(const QrMat *mats, int32_t b, const void *a_, void *ws_) {
  using T = typename ElemOf<C>::T;
  constexpr int TH = 64 * NW;
  constexpr int kStageCols = C ? 4 : 8;   // panel columns staged together between memory and registers
  constexpr size_t kApplyBytes = sizeof(T) * (NW + 2) * kNB * (kNB + 1);
  constexpr size_t kStageBytes = sizeof(T) * TH * (kStageCols + 1);
  __shared__ __align__(16) char smem[kApplyBytes > kStageBytes ? kApplyBytes : kStageBytes];
  __shared__ T sSum[2][NW][kNB], sRow[2][kNB], sV[kNB][kNB + 1], sTau[kNB];
  const QrMat mt = mats[blockIdx.x];
  const int64_t m = mt.m, n = mt.n, k = mt.k;
  const int64_t tile = FIRST ? int64_t(blockIdx.y) : int64_t(b) + 1 + blockIdx.y;
  const int64_t j0 = tile * kNB;
  if (j0 >= n || int64_t(b) * kNB >= k) return;
  const int nc = static_cast<int>(n - j0 < kNB ? n - j0 : kNB);
  T *W = static_cast<T *>(ws_) + mt.w_off;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const T *src = W;
  if constexpr (FIRST) {
    const T *A = static_cast<const T *>(a_) + mt.a_off;
    if (tile != 0) {
      const int c = tid % kNB;
      if (c < nc)
        for (int64_t i = tid / kNB; i < m; i += TH / kNB) W[i * n + j0 + c] = A[i * n + j0 + c];
      return;
    }
    src = A;
  } else {
    auto *sPart = reinterpret_cast<T (*)[kNB][kNB + 1]>(smem);
    apply_block<C, NW, true, PAD>(static_cast<const T *>(ws_) + mt.v_off + int64_t(b) * m * kNB, v_cols<PAD>(k, b),
                             static_cast<const T *>(ws_) + mt.t_off + int64_t(b) * kNB * kNB, W + j0, n,
                             int64_t(b) * kNB, m, nc, sPart, sPart[NW], sPart[NW + 1]);
    if (tile != int64_t(b) + 1 || j0 >= k) return;
  }
  __syncthreads();

  // ---- the panel: local row tid + TH r in registers, columns 0 .. kNB - 1 ----
  // A wave's 64 rows pass through LDS so that memory is read and written in
  // runs of kStageCols elements.
  const int64_t mp = m - j0;
  const int kc = block_cols(k, tile);
  T x[kNB][RPT];
  auto *sStage = reinterpret_cast<T (*)[kStageCols + 1]>(smem) + 64 * w;
  constexpr int kRowsPerLoad = 64 / kStageCols;
  const int scol = lane % kStageCols, srow = lane / kStageCols;
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int64_t base = 64 * w + int64_t(TH) * r;
#pragma unroll
    for (int c0 = 0; c0 < kNB; c0 += kStageCols) {
#pragma unroll
      for (int q = 0; q < 64; q += kRowsPerLoad) {
        const int64_t i = base + q + srow;
        const bool ok = i < mp && c0 + scol < nc;
        sStage[q + srow][scol] = ok ? src[(j0 + i) * n + j0 + c0 + scol] : zero_<T>();
      }
      wave_lds_sync();
#pragma unroll
      for (int s = 0; s < kStageCols; ++s) x[c0 + s][r] = sStage[lane][s];
      wave_lds_sync();
    }
  }
  // At step c slot s holds column (c + s) mod kNB: the slots turn by one per
  // step, so that registers are indexed by constants only.
#pragma unroll 1
  for (int c = 0; c < kNB; ++c) {
    const int buf = c & 1;
    T d[kNB];
#pragma unroll
    for (int s = 0; s < kNB; ++s) d[s] = zero_<T>();
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const T xi = sel_(r > 0 || tid > c, x[0][r], zero_<T>());
#pragma unroll
      for (int s = 0; s < kNB; ++s) d[s] = add_(d[s], cmul_(xi, x[s][r]));
    }
    const T part = wave_sums16(d, lane);
    if ((lane & 3) == 0) sSum[buf][w][lane >> 2] = part;
    if (tid == c) {
#pragma unroll
      for (int s = 0; s < kNB; ++s) sRow[buf][s] = x[s][0];
    }
    __syncthreads();
    // every wave: slot s in lane s (and its copies s + 16, ...)
    const int s_ = lane & (kNB - 1);
    T tot = sSum[buf][0][s_];
#pragma unroll
    for (int g = 1; g < NW; ++g) tot = add_(tot, sSum[buf][g][s_]);
    const T row = sRow[buf][s_];
    const T alpha = lane_value(row, 0);
    const double xn2 = re_(lane_value(tot, 0));
    const double ai = C ? (abs2_(alpha) - re_(alpha) * re_(alpha)) : 0.0;   // (Im alpha)^2
    T t = zero_<T>(), sc = zero_<T>(), bt = alpha;
    if (c < kc && !(xn2 == 0.0 && ai == 0.0)) {
      const double nrm = sqrt(abs2_(alpha) + xn2);
      const double beta = re_(alpha) >= 0.0 ? -nrm : nrm;
      bt = scl_(beta, one_<T>());
      t = scl_(1.0 / beta, sub_(bt, alpha));
      sc = recip_(sub_(alpha, bt));
    }
    // column j = c + s: v^H x_j = x_cj + conj(sc) sum; earlier column j:
    // v_j^H v = sc conj(sum) + conj(v_cj), kept for T
    const T f = mul_(conj_(t), add_(row, mul_(conj_(sc), tot)));
    if (w == 0 && lane < kNB && lane >= kNB - c) sV[c][c + lane - kNB] = add_(mul_(sc, conj_(tot)), conj_(row));
    if (tid == 0) sTau[c] = t;
    T vi[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r)
      vi[r] = sel_(r > 0 || tid > c, mul_(sc, x[0][r]), sel_(tid == c, one_<T>(), zero_<T>()));
    if (abs2_(t) != 0.0) {
#pragma unroll
      for (int s = 1; s < kNB; ++s) {
        if (s < kNB - c) {
          const T fs = lane_value(f, s);
#pragma unroll
          for (int r = 0; r < RPT; ++r) x[s][r] = sub_(x[s][r], mul_(vi[r], fs));
        }
      }
    }
    T cur[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      // a column past the last reflector keeps its R entries
      cur[r] = sel_(c >= kc, x[0][r], sel_(r > 0 || tid > c, vi[r], sel_(tid == c, bt, x[0][r])));
    }
#pragma unroll
    for (int s = 0; s + 1 < kNB; ++s)
#pragma unroll
      for (int r = 0; r < RPT; ++r) x[s][r] = x[s + 1][r];
#pragma unroll
    for (int r = 0; r < RPT; ++r) x[kNB - 1][r] = cur[r];
  }

  // ---- R rows of the panel, the reflectors, T ----
  if (tid < kNB && tid < mp) {
#pragma unroll
    for (int s = 0; s < kNB; ++s)
      if (s >= tid && s < nc) W[(j0 + tid) * n + j0 + s] = x[s][0];
  }
  const int64_t pb = FIRST ? 0 : int64_t(b) + 1;
  T *V = static_cast<T *>(ws_) + mt.v_off + pb * m * kNB;
  const int ldv = v_cols<PAD>(k, pb);
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int64_t base = 64 * w + int64_t(TH) * r;
#pragma unroll
    for (int c0 = 0; c0 < kNB; c0 += kStageCols) {
#pragma unroll
      for (int s = 0; s < kStageCols; ++s) {
        const int c = c0 + s;
        const bool below = r > 0 || tid > c;
        sStage[lane][s] = sel_(c < kc && below, x[c][r], sel_(c < kc && r == 0 && tid == c, one_<T>(), zero_<T>()));
      }
      wave_lds_sync();
#pragma unroll
      for (int q = 0; q < 64; q += kRowsPerLoad) {
        const int64_t i = base + q + srow;
        if (i < mp && (PAD || c0 + scol < kc)) V[(j0 + i) * ldv + c0 + scol] = sStage[q + srow][scol];
      }
      wave_lds_sync();
    }
  }
  __syncthreads();
  // T by columns: T[:c, c] = -tau_c T[:c, :c] (V^H v_c), T[c, c] = tau_c; lane
  // j keeps row j
  if (w == 0 && lane < kNB) {
    T trow[kNB];
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      T s = zero_<T>();
#pragma unroll
      for (int l = 0; l < c; ++l) s = add_(s, sel_(l >= lane, mul_(trow[l], sV[c][l]), zero_<T>()));
      const T tau = sTau[c];
      const T e = mul_(tau, s);
      trow[c] = sel_(lane < c, sub_(zero_<T>(), e), sel_(lane == c, tau, zero_<T>()));
    }
    T *Tm = static_cast<T *>(ws_) + mt.t_off + pb * kNB * kNB;
#pragma unroll
    for (int c = 0; c < kNB; ++c) Tm[lane * kNB + c] = trow[c];
  }
}

// R and Q, grid (matrices, column tiles): columns j0 .. of R, and the same
// columns of Q = H_0 ... H_{k-1} I, the blocks applied from the tile's own
// one back to the first (a later block acts on rows where the tile is zero).
template <bool C, int NW, bool PAD>
__global__ void __launch_bounds__(64 * NW) k_qr_q(const QrMat *mats, const void *ws_, void *q_, void *r_) {
  using T = typename ElemOf<C>::T;
  constexpr int TH = 64 * NW;
  __shared__ T sPart[NW + 2][kNB][kNB + 1];
  const QrMat mt = mats[blockIdx.x];
  const int64_t m = mt.m, n = mt.n, k = mt.k;
  const int64_t j0 = int64_t(blockIdx.y) * kNB;
  if (j0 >= n) return;
  const int c = threadIdx.x % kNB;
  const T *W = static_cast<const T *>(ws_) + mt.w_off;
  T *R = static_cast<T *>(r_) + mt.r_off;
  T *Q = static_cast<T *>(q_) + mt.q_off;
  if (j0 + c < n)
    for (int64_t i = threadIdx.x / kNB; i < k; i += TH / kNB)
      R[i * n + j0 + c] = j0 + c >= i ? W[i * n + j0 + c] : zero_<T>();
  if (j0 >= k) return;
  if (j0 + c < k)
    for (int64_t i = threadIdx.x / kNB; i < m; i += TH / kNB) Q[i * k + j0 + c] = i == j0 + c ? one_<T>() : zero_<T>();
  const int nc = static_cast<int>(k - j0 < kNB ? k - j0 : kNB);
  for (int64_t b = blockIdx.y; b >= 0; --b) {
    __syncthreads();
    apply_block<C, NW, false, PAD>(static_cast<const T *>(ws_) + mt.v_off + b * m * kNB, v_cols<PAD>(k, b),
                              static_cast<const T *>(ws_) + mt.t_off + b * kNB * kNB, Q + j0, k, b * kNB, m, nc, sPart,
                              sPart[NW], sPart[NW + 1]);
  }
}

// Matrices with more rows than a panel in registers takes, and small ones: one
// workgroup per matrix, unblocked.
template <typename T>
__device__ __forceinline__ double block_sum(double v, double *red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const double s = red[0] + red[1] + red[2] + red[3];
  __syncthreads();
  return s;
}

template <bool C>
__global__ void __launch_bounds__(kThreads) k_qr_generic(const QrMat *mats, const void *a_, void *ws_, void *q_, void *r_) {
  using T = typename ElemOf<C>::T;
  __shared__ double sRed[kWaves];
  __shared__ T sTau, sScale;
  const QrMat mt = mats[blockIdx.x];
  const T *A = static_cast<const T *>(a_) + mt.a_off;
  T *Wm = static_cast<T *>(ws_) + mt.w_off;
  T *Qw = static_cast<T *>(ws_) + mt.v_off;
  T *tau = static_cast<T *>(ws_) + mt.t_off;
  const int64_t m = mt.m, n = mt.n, k = mt.k;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int64_t e = threadIdx.x; e < m * n; e += kThreads) {
    const int64_t j = e / m, i = e - j * m;
    Wm[e] = A[i * n + j];
  }
  __syncthreads();
  for (int64_t j = 0; j < k; ++j) {
    T *col = Wm + j * m;
    double part = 0.0;
    for (int64_t i = j + 1 + threadIdx.x; i < m; i += kThreads) part += abs2_(col[i]);
    const double xn2 = block_sum<T>(part, sRed);
    if (threadIdx.x == 0) {
      const T alpha = col[j];
      T t = zero_<T>(), sc = zero_<T>();
      const double ai = C ? (abs2_(alpha) - re_(alpha) * re_(alpha)) : 0.0;   // (Im alpha)^2
      if (!(xn2 == 0.0 && ai == 0.0)) {
        const double nrm = sqrt(abs2_(alpha) + xn2);
        const double beta = re_(alpha) >= 0.0 ? -nrm : nrm;
        T bt = zero_<T>();
        bt = add_(bt, scl_(beta, one_<T>()));
        t = scl_(1.0 / beta, sub_(bt, alpha));
        sc = recip_(sub_(alpha, bt));
        col[j] = bt;
      }
      sTau = t;
      sScale = sc;
      tau[j] = t;
    }
    __syncthreads();
    const T t = sTau;
    if (abs2_(t) == 0.0) continue;
    const T sc = sScale;
    for (int64_t i = j + 1 + threadIdx.x; i < m; i += kThreads) col[i] = mul_(sc, col[i]);
    __syncthreads();
    // trailing columns: x <- H^H x = x - conj(tau) v (v^H x)
    const T ct = conj_(t);
    for (int64_t c = j + 1 + wave; c < n; c += kWaves) {
      T *x = Wm + c * m;
      T d = zero_<T>();
      for (int64_t i = j + lane; i < m; i += 64) {
        const T vi = (i == j) ? one_<T>() : col[i];
        d = add_(d, cmul_(vi, x[i]));
      }
      if constexpr (C) {
        d.x = wave_sum(d.x);
        d.y = wave_sum(d.y);
      } else {
        d = wave_sum(d);
      }
      const T f = mul_(ct, d);
      for (int64_t i = j + lane; i < m; i += 64) {
        const T vi = (i == j) ? one_<T>() : col[i];
        x[i] = sub_(x[i], mul_(vi, f));
      }
    }
    __syncthreads();
  }
  // R (k x n), upper triangle of W
  T *R = static_cast<T *>(r_) + mt.r_off;
  for (int64_t e = threadIdx.x; e < k * n; e += kThreads) {
    const int64_t i = e / n, c = e - i * n;
    R[e] = c >= i ? Wm[c * m + i] : zero_<T>();
  }
  // Q = H_0 ... H_{k-1} I[:, :k]
  for (int64_t e = threadIdx.x; e < m * k; e += kThreads) {
    const int64_t c = e / m, i = e - c * m;
    Qw[e] = (i == c) ? one_<T>() : zero_<T>();
  }
  __syncthreads();
  for (int64_t j = k - 1; j >= 0; --j) {
    const T t = tau[j];
    if (abs2_(t) == 0.0) continue;
    const T *v = Wm + j * m;
    for (int64_t c = j + wave; c < k; c += kWaves) {
      T *x = Qw + c * m;
      T d = zero_<T>();
      for (int64_t i = j + lane; i < m; i += 64) {
        const T vi = (i == j) ? one_<T>() : v[i];
        d = add_(d, cmul_(vi, x[i]));
      }
      if constexpr (C) {
        d.x = wave_sum(d.x);
        d.y = wave_sum(d.y);
      } else {
        d = wave_sum(d);
      }
      const T f = mul_(t, d);
      for (int64_t i = j + lane; i < m; i += 64) {
        const T vi = (i == j) ? one_<T>() : v[i];
        x[i] = sub_(x[i], mul_(vi, f));
      }
    }
    __syncthreads();
  }
  T *Q = static_cast<T *>(q_) + mt.q_off;
  for (int64_t e = threadIdx.x; e < m * k; e += kThreads) {
    const int64_t i = e / k, c = e - i * k;
    Q[e] = Qw[c * m + i];
  }
}

// Rows a panel takes: 512 threads of 4 (FP64) or 3 (complex) rows.  Three complex
// rows do not fit the 256 registers of a thread (111 spill to scratch): 1025 to 1536
// complex rows run slower than the registers would allow, and still faster than
// unblocked (one 1200 x 600 matrix 813 -> 6.2 ms, one of 1025 x 17 561 -> 333 us).
template <bool C>
constexpr int64_t kMaxBlockedRows = C ? 1536 : 2048;

// Small matrices go to k_qr_generic when the whole call is of them, or when they
// are many: one workgroup walks their few short columns faster than the launches of
// the blocked form come and go, and more of them fit a compute unit (us, generic |
// blocked: one 2 x 2 FP64 28 | 44, one 8 x 8 45 | 45, one 4 x 64 57 | 48, one 1024 x 4
// 75 | 68; 3000 of 4 x 4 65 | 185, of 12 x 12 184 | 198, of 16 x 16 251 | 205, of
// 1500 x 1 468 | 908, of 256 x 8 603 | 476; complex128, one 10 x 10 58 | 62, one
// 1024 x 4 80 | 102, 300 of 12 x 12 81 | 111, of 8 x 64 166 | 131, 1000 of 16 x 16
// 159 | 186, 3000 of 24 x 24 615 | 1075, of 32 x 32 1248 | 1096).  A few among larger
// ones are not worth a launch of their own (about 30 us).
template <bool C>
constexpr int64_t kManySmall = C ? 256 : 512;
template <bool C>
bool small_matrix(int64_t m, int64_t n, int64_t k, int64_t n_mats) {
  if (C && n_mats >= 512 && m <= 24 && n <= 24) return true;
  if (k > 24 || m * k * k > (C ? 16384 : 9216)) return false;
  if (n_mats < kManySmall<C>) return n <= (C ? 128 : 512) && k * k * n <= (C ? 1000 : 512);
  return k * k * n <= (C ? 2048 : 1800);
}

template <bool C>
qlt_status qr_impl(int64_t n_mats, const int64_t *rows, const int64_t *cols, const void *a, const int64_t *a_offsets,
                   void *q, const int64_t *q_offsets, void *r, const int64_t *r_offsets, hipStream_t st) {
  const size_t esz = C ? 16 : 8;
  int64_t n_small = 0;
  for (int64_t i = 0; i < n_mats; ++i) n_small += small_matrix<C>(rows[i], cols[i], std::min(rows[i], cols[i]), n_mats);
  const bool all_small = n_small == n_mats, small_apart = all_small || n_small >= kManySmall<C>;
  const auto is_blocked = [&](int64_t m, int64_t n, int64_t k) {
    return !all_small && m <= kMaxBlockedRows<C> && (n + kNB - 1) / kNB <= 65535 &&
           !(small_apart && small_matrix<C>(m, n, k, n_mats));
  };
  int64_t n_blocked = 0, compact = 0, padding = 0;   // elements of scratch
  for (int64_t i = 0; i < n_mats && !all_small; ++i) {
    const int64_t m = rows[i], n = cols[i], k = std::min(m, n);
    compact += m * (n + k);
    if (!is_blocked(m, n, k)) continue;
    ++n_blocked;
    padding += m * ((k + kNB - 1) / kNB * kNB - k);
  }
  const bool pad = padding <= compact / 4;
  // the blocked matrices, then k_qr_generic's
  std::vector<QrMat> mats(static_cast<size_t>(n_mats));
  int64_t ws = 0, max_rows = 0, max_blocks = 0, max_tiles = 0, at_blocked = 0, at_generic = n_blocked;
  for (int64_t i = 0; i < n_mats; ++i) {
    const bool blocked = is_blocked(rows[i], cols[i], std::min(rows[i], cols[i]));
    QrMat &mt = mats[static_cast<size_t>(blocked ? at_blocked++ : at_generic++)];
    mt.m = rows[i];
    mt.n = cols[i];
    mt.k = std::min(rows[i], cols[i]);
    const int64_t nb = (mt.k + kNB - 1) / kNB;
    mt.w_off = ws;
    ws += mt.m * mt.n;
    mt.v_off = ws;
    ws += mt.m * (blocked && pad ? nb * kNB : mt.k);
    mt.t_off = ws;
    ws += blocked ? nb * kNB * kNB : mt.k;
    mt.a_off = a_offsets[i];
    mt.q_off = q_offsets[i];
    mt.r_off = r_offsets[i];
    if (blocked) {
      max_rows = std::max(max_rows, mt.m);
      max_blocks = std::max(max_blocks, nb);
      max_tiles = std::max(max_tiles, (mt.n + kNB - 1) / kNB);
    }
  }
  DevBuf d_ws, d_mats;
  QLT_HIP(hipMalloc(&d_ws.p, std::max<size_t>(1, static_cast<size_t>(ws) * esz)));
  QLT_HIP(hipMalloc(&d_mats.p, sizeof(QrMat) * mats.size()));
  QLT_HIP(hipMemcpyAsync(d_mats.p, mats.data(), sizeof(QrMat) * mats.size(), hipMemcpyHostToDevice, st));
  const auto *dm = static_cast<const QrMat *>(d_mats.p);
  const unsigned gm = static_cast<unsigned>(n_blocked);
  if (n_blocked < n_mats)
    hipLaunchKernelGGL(k_qr_generic<C>, dim3(static_cast<unsigned>(n_mats - n_blocked)), dim3(kThreads), 0, st,
                       dm + n_blocked, a, d_ws.p, q, r);
  auto launch_pad = [&](auto nw_tag, auto rpt_tag, auto pad_tag) {
    constexpr int NW = decltype(nw_tag)::value, RPT = decltype(rpt_tag)::value;
    constexpr bool PAD = decltype(pad_tag)::value;
    hipLaunchKernelGGL((k_qr_step<C, NW, RPT, true, PAD>), dim3(gm, static_cast<unsigned>(max_tiles)), dim3(64 * NW), 0, st,
                       dm, -1, a, d_ws.p);
    for (int64_t b = 0; b + 1 < max_tiles && b < max_blocks; ++b)
      hipLaunchKernelGGL((k_qr_step<C, NW, RPT, false, PAD>), dim3(gm, static_cast<unsigned>(max_tiles - b - 1)),
                         dim3(64 * NW), 0, st, dm, static_cast<int32_t>(b), a, d_ws.p);
    hipLaunchKernelGGL((k_qr_q<C, 4, PAD>), dim3(gm, static_cast<unsigned>(max_tiles)), dim3(256), 0, st, dm, d_ws.p, q,
                       r);
  };
  auto launch = [&](auto nw_tag, auto rpt_tag) {
    if (pad) launch_pad(nw_tag, rpt_tag, std::true_type{});
    else launch_pad(nw_tag, rpt_tag, std::false_type{});
  };
  using std::integral_constant;
  if (max_tiles > 0) {
    // the fewest waves whose registers hold the tallest panel: a column costs
    // every wave its own reduction
    if (max_rows <= 512) launch(integral_constant<int, 4>{}, integral_constant<int, 2>{});
    else if (max_rows <= 1024) launch(integral_constant<int, 8>{}, integral_constant<int, 2>{});
    else launch(integral_constant<int, 8>{}, integral_constant<int, C ? 3 : 4>{});
  }
  QLT_HIP(hipGetLastError());
  QLT_HIP(hipStreamSynchronize(st));
  return QLT_OK;
}

}  // namespace

extern "C" {

qlt_status qlt_block_qr(int32_t dtype, int64_t n_mats, const int64_t *rows, const int64_t *cols, const void *a,
                        const int64_t *a_offsets, void *q, const int64_t *q_offsets, void *r,
                        const int64_t *r_offsets, void *stream) {
  QLT_REQUIRE_INIT();
  QLT_CHECK_ARG(qlt::valid_dtype(dtype), "qlt_block_qr: bad dtype");
  QLT_TRY(check_shapes("qlt_block_qr", n_mats, rows, cols));
  if (n_mats == 0) return QLT_OK;
  QLT_CHECK_ARG(a != nullptr && q != nullptr && r != nullptr, "qlt_block_qr: null data pointer");
  QLT_CHECK_ARG(a_offsets != nullptr && q_offsets != nullptr && r_offsets != nullptr,
                "qlt_block_qr: null offset array");
  QLT_CHECK_ARG(!qlt::stream_capturing(qlt::as_stream(stream)), "qlt_block_qr: not capturable (allocates)");
  if (qlt::dtype_is_single(dtype)) {
    const int32_t wide = dtype == QLT_F32 ? QLT_F64 : QLT_C128;
    const int64_t esz = qlt::dtype_bytes(wide);
    std::vector<int64_t> kk(static_cast<size_t>(n_mats));
    for (int64_t i = 0; i < n_mats; ++i) kk[i] = std::min(rows[i], cols[i]);
    const int64_t na = extent(n_mats, a_offsets, rows, cols);
    const int64_t nq = extent(n_mats, q_offsets, rows, kk.data());
    const int64_t nr = extent(n_mats, r_offsets, kk.data(), cols);
    DevBuf wa, wq, wr;
    QLT_HIP(hipMalloc(&wa.p, std::max<int64_t>(1, na) * esz));
    QLT_HIP(hipMalloc(&wq.p, std::max<int64_t>(1, nq) * esz));
    QLT_HIP(hipMalloc(&wr.p, std::max<int64_t>(1, nr) * esz));
    QLT_TRY(qlt_convert(dtype, wide, na, a, wa.p, stream));
    QLT_TRY(qlt_block_qr(wide, n_mats, rows, cols, wa.p, a_offsets, wq.p, q_offsets, wr.p, r_offsets, stream));
    QLT_TRY(qlt_convert(wide, dtype, nq, wq.p, q, stream));
    QLT_TRY(qlt_convert(wide, dtype, nr, wr.p, r, stream));
    QLT_HIP(hipStreamSynchronize(qlt::as_stream(stream)));
    return QLT_OK;
  }
  if (dtype == QLT_F64)
    return qr_impl<false>(n_mats, rows, cols, a, a_offsets, q, q_offsets, r, r_offsets, qlt::as_stream(stream));
  return qr_impl<true>(n_mats, rows, cols, a, a_offsets, q, q_offsets, r, r_offsets, qlt::as_stream(stream));
}

}  // extern "C"
