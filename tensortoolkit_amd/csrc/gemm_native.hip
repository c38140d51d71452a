// Grouped block GEMM over a contraction plan, native FP64 / complex128 MFMA.
//
// Replaces the execution loop of CtrctTwoBSDTAndAssignIn
// (include/qlten/qltensor/blk_spar_data_ten/global_operations.h:895-992):
// there, every task lazily transposes its A and B blocks with HPTT/cuTENSOR
// (hp_numeric::TensorTranspose, framework/hp_numeric/ten_trans.h:56-114,245-349)
// and then issues one BLAS call C_blk = A'(m x k) B'(k x n) + beta C_blk
// (hp_numeric::MatMultiply, framework/hp_numeric/blas_level3.h:35-56,798-856).
// Here one launch covers the whole plan (k_all_classes).  Each workgroup owns
// one TM x TN tile (64 or 32 each way; 32 x 16 for n <= 16) of one output
// block, or one k-slice of it, and walks every task of that block, so the
// per-block beta chain (0 for the first task, 1 after) becomes a single write
// of the finished tile (or of its slices' sum).  Outputs of n <= 4 go to a
// row-streaming path, or to row panels.  The transposes are never
// materialised: the prologue gathers A'(i, p) = A[a_off + row_off(i) + col_off(p)] straight
// from the original block layout through per-tile offset tables, staging the
// k-chunk in LDS, with the thread mapping chosen so that the block's
// innermost memory axis is read contiguously.

#include <algorithm>
#include <cstdio>
#include <memory>
#include <type_traits>

#include "qlt_internal.h"

using namespace qlt;

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

// Element access of the raw data: E is the stored real type (double, or
// float for QLTEN_Float / QLTEN_ComplexFloat tensors), complex elements are
// interleaved (re, im); arithmetic is FP64 either way.  `p` points to the
// element (its real part).
template <typename E, bool CPLX>
__device__ __forceinline__ double2 ld_elem(const E *p) {
  if constexpr (CPLX) {
    if constexpr (sizeof(E) == 8) {
      return *reinterpret_cast<const double2 *>(p);
    } else {
      const float2 f = *reinterpret_cast<const float2 *>(p);
      return double2{static_cast<double>(f.x), static_cast<double>(f.y)};
    }
  } else {
    return double2{static_cast<double>(*p), 0.0};
  }
}
// The same load with the non-temporal hint, for streams read exactly once
// (FP64 storage; the single-precision types take the plain load).
template <typename E, bool CPLX>
__device__ __forceinline__ double2 ld_elem_stream(const E *p) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  if constexpr (CPLX && sizeof(E) == 8) {
    const v2d v = __builtin_nontemporal_load(reinterpret_cast<const v2d *>(p));
    return double2{v[0], v[1]};
  } else if constexpr (!CPLX && sizeof(E) == 8) {
    return double2{__builtin_nontemporal_load(reinterpret_cast<const double *>(p)), 0.0};
  } else {
    return ld_elem<E, CPLX>(p);
  }
}
// The stored form of one element as it sits in registers between its load and
// its LDS staging: double2 / float2 (complex), double / float (real).  The
// GEMM fetches keep this form and convert to FP64 only when staging, so a
// single-precision load is not followed by a conversion inside its guard,
// which would make every load wait for its data before the next one issues.
template <typename E, bool CPLX>
using raw_t = std::conditional_t<CPLX, std::conditional_t<sizeof(E) == 8, double2, float2>, E>;
template <typename E, bool CPLX>
__device__ __forceinline__ raw_t<E, CPLX> ld_raw(const E *p) {
  return *reinterpret_cast<const raw_t<E, CPLX> *>(p);
}
__device__ __forceinline__ double re_of(double2 v) { return v.x; }
__device__ __forceinline__ double re_of(float2 v) { return static_cast<double>(v.x); }
__device__ __forceinline__ double re_of(double v) { return v; }
__device__ __forceinline__ double re_of(float v) { return static_cast<double>(v); }
__device__ __forceinline__ double im_of(double2 v) { return v.y; }
__device__ __forceinline__ double im_of(float2 v) { return static_cast<double>(v.y); }
__device__ __forceinline__ double im_of(double) { return 0.0; }
__device__ __forceinline__ double im_of(float) { return 0.0; }
template <typename E, bool CPLX>
__device__ __forceinline__ void zero_unless(raw_t<E, CPLX> &v, bool ok) {
  if constexpr (CPLX) {
    v.x = ok ? v.x : E(0);
    v.y = ok ? v.y : E(0);
  } else {
    v = ok ? v : E(0);
  }
}
template <typename E, bool CPLX>
__device__ __forceinline__ void st_elem(E *p, double re, double im) {
  if constexpr (CPLX) {
    if constexpr (sizeof(E) == 8) *reinterpret_cast<double2 *>(p) = double2{re, im};
    else *reinterpret_cast<float2 *>(p) = float2{static_cast<float>(re), static_cast<float>(im)};
  } else {
    *p = static_cast<E>(re);
  }
}

// Offset of a linear index inside a block over one part's axes (split_offset),
// with the descriptor's numbers read once per task: up to two axes take one
// multiply-shift division and no further reads, more take the loop, whose
// scalar reads of every axis are waited for at every element (they were most
// of a step of a contraction not affine in k: a U(1) chi = 40 pair of rank-4
// tensors over cyclic axes, complex64, 99 -> 51 us, FP64 79 -> 38 us).  The row
// class, where 16 threads take the offsets of a step, keeps the plain form: these
// numbers cost it 16 registers and a wave per SIMD.
struct PartSplit {
  const BlkGather *g;
  int n;
  uint64_t mag;      // of the inner of two axes; 0: one axis
  int32_t sh, dim, outer, inner;
};
template <bool ROW>
__device__ __forceinline__ PartSplit part_split(const BlkGather &g, int n) {
  PartSplit p{&g, n, 0, 0, 1, 0, 0};
  const int32_t *strs = ROW ? g.rstr : g.cstr;
  if (n == 1) {
    p.inner = strs[0];
  } else if (n == 2) {
    p.mag = ROW ? g.rmag[1] : g.cmag[1];
    p.sh = ROW ? g.rsh[1] : g.csh[1];
    p.dim = ROW ? g.rdim[1] : g.cdim[1];
    p.outer = strs[0];
    p.inner = strs[1];
  }
  return p;
}
template <bool ROW>
__device__ __forceinline__ int32_t offset_of(const PartSplit &p, int32_t x) {
  if (p.n > 2)
    return ROW ? split_offset(x, p.g->rdim, p.g->rstr, p.g->rmag, p.g->rsh, p.n)
               : split_offset(x, p.g->cdim, p.g->cstr, p.g->cmag, p.g->csh, p.n);
  const int32_t q = static_cast<int32_t>((static_cast<uint64_t>(x) * p.mag) >> p.sh);
  return q * p.outer + (x - q * p.dim) * p.inner;
}

// Epilogue of one output element: C = alpha * x + beta * old, with `old` the
// element's earlier value, loaded by the caller beforehand (not read when
// beta == 0).  The epilogues load every old value of a thread first, at
// addresses clamped into the block, so the loads are in flight together
// rather than each waited on before its store.
template <typename E, bool CPLX>
__device__ __forceinline__ void st_scaled(E *cp, double xr, double xi, const raw_t<E, CPLX> &old, bool use_beta,
                                          double alpha_r, double alpha_i, double beta_r, double beta_i) {
  if constexpr (CPLX) {
    double yr = alpha_r * xr - alpha_i * xi, yi = alpha_r * xi + alpha_i * xr;
    if (use_beta) {
      const double o_r = re_of(old), o_i = im_of(old);
      yr += beta_r * o_r - beta_i * o_i;
      yi += beta_r * o_i + beta_i * o_r;
    }
    st_elem<E, true>(cp, yr, yi);
  } else {
    double y = alpha_r * xr;
    if (use_beta) y += beta_r * re_of(old);
    st_elem<E, false>(cp, y, 0.0);
  }
}

// Epilogue of an MFMA output tile: element (mt, nt, v) of a thread sits at
// row r0 + 16 mt + 4 v, column c0 + 16 nt.  With beta == 0 the stores go out
// back to back; otherwise every old value is loaded first (addresses clamped
// to the block's first element) and the stores follow.  The two cases are
// separate code: merged, the waits for the loads would also hold back the
// stores of the beta == 0 case, since stores count in the same counter.
// ACC is one 16 x 16 sub-tile's 4 values of a thread (v4d, or double[4]).
template <bool CPLX, int BM, int BN, typename E, typename ACC>
__device__ __forceinline__ void tile_epilogue(const Seg &seg, int r0, int c0, const ACC (&acc)[BM][BN],
                                              const ACC (&acc_i)[BM][BN], E *__restrict__ C, double alpha_r,
                                              double alpha_i, double beta_r, double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  auto store_all = [&](auto with_beta, const raw_t<E, CPLX>(&old)[BM][BN][4]) {
    constexpr bool WB = decltype(with_beta)::value;
#pragma unroll
    for (int mt = 0; mt < BM; ++mt)
#pragma unroll
      for (int nt = 0; nt < BN; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + mt * 16 + 4 * v, col = c0 + nt * 16;
          if (row < seg.m && col < seg.n) {
            const int64_t idx = seg.c_off + static_cast<int64_t>(row) * seg.n + col;
            st_scaled<E, CPLX>(C + P * idx, acc[mt][nt][v], CPLX ? acc_i[mt][nt][v] : 0.0, old[mt][nt][v], WB,
                               alpha_r, alpha_i, beta_r, beta_i);
          }
        }
  };
  if (beta_r != 0.0 || beta_i != 0.0) {
    raw_t<E, CPLX> old[BM][BN][4];
#pragma unroll
    for (int mt = 0; mt < BM; ++mt)
#pragma unroll
      for (int nt = 0; nt < BN; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + mt * 16 + 4 * v, col = c0 + nt * 16;
          const bool ok = row < seg.m && col < seg.n;
          old[mt][nt][v] = ld_raw<E, CPLX>(C + P * (seg.c_off + (ok ? static_cast<int64_t>(row) * seg.n + col : 0)));
        }
    store_all(std::true_type{}, old);
  } else {
    const raw_t<E, CPLX> none[BM][BN][4] = {};
    store_all(std::false_type{}, none);
  }
}

constexpr int KC = kKChunk;   // plan step: k-chunk of 16
constexpr double kPanelStreamBytes = 256.0 * 1024 * 1024;   // the MI355X last-level (Infinity) cache

// Tile order for the XCDs: workgroups are dispatched to the 8 XCDs round
// robin, so workgroup b runs on XCD b % 8.  Mapping b to logical tile
// (r / G) * 8G + (b % 8) * G + r % G, with r = b / 8, gives each XCD runs of G
// consecutive tiles (neighbouring tiles of one output block, which share A
// rows or B columns) while keeping the global longest-first order at a
// granularity of 8G tiles; the tail beyond the last full 8G group maps to
// itself.
constexpr int kXcds = 8;
constexpr int kXcdRun = 4;
__device__ __forceinline__ int xcd_tile(int b, int n) {
  constexpr int span = kXcds * kXcdRun;
  if (b >= (n / span) * span) return b;
  const int r = b / kXcds;
  return (r / kXcdRun) * span + (b % kXcds) * kXcdRun + (r % kXcdRun);
}

// Grouped MFMA kernel, one 256-thread workgroup per TM x TN output tile
// (TM, TN in {32, 64}); the four waves split the tile 2 x 2, each wave
// computing (TM/2) x (TN/2) as BM x BN blocks of v_mfma_f64_16x16x4f64.
//   What bounds it: the MFMAs are busy about half of the time (64 cycles each;
// 45 us of a 100 us D = 2048 FP64 launch), the rest is the chain of a step --
// loads, LDS, barrier -- that three to five workgroups per CU only partly
// cover.  Measured without gain: loads issued two steps ahead (249 us either
// way at D = 2048 FP64), 8-deep complex steps at four workgroups per CU (1.14
// ms either way at D = 4096), B' fragments loaded past LDS (249 -> 308 us), and
// 64 x 64 tiles (303 -> 376 us).
// The staged chunk, real and imaginary planes, in one buffer (the next chunk
// waits in registers): with two a step takes one barrier less, but twice the LDS,
// and was slower at the same number of workgroups per CU (D = 2048 FP64 matvec 255
// -> 246 us with its data in the cache, D = 4096 complex128 1.146 -> 1.119 ms; at
// four complex workgroups per CU, which one buffer leaves room for, the registers
// spill: 1.139 ms).  A' by rows (18 doubles apart), B' by k (TN + 4 doubles apart),
// contracted index p at place k_place(p).  Lane (lr, lk) finds the indices lk, 4 + lk, 8 + lk, 12 + lk of the four
// MFMA steps at places 4 lk .. 4 lk + 3: A' is read in 16-byte pieces, and both
// strides keep a wave's reads and the k-contiguous / n-contiguous writes free
// of bank conflicts (with both operands by k and rows one double more than a
// power of two apart, every read took two passes: D = 2048 FP64 matvec 308 ->
// 277 us).
__device__ __forceinline__ int k_place(int p) { return ((p & 3) << 2) | (p >> 2); }
template <bool CPLX, int TMv, int TNv>
struct GroupedShared {
  static constexpr int P = CPLX ? 2 : 1;
  double As[P][TMv][KC + 2];
  double Bs[P][KC][TNv + 4];
};
template <bool CPLX, int TMv, int TNv, typename E>
__device__ __forceinline__ void grouped_tile(
    char *smem, const Tile tile, const Seg *__restrict__ segs, const ExecTask *__restrict__ exec,
    const BlkGather *__restrict__ ga, const BlkGather *__restrict__ gb, const GatherLayout &L,
    const E *__restrict__ A, const E *__restrict__ B, E *__restrict__ C, double *__restrict__ part,
    double alpha_r, double alpha_i, double beta_r, double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  constexpr int QA = TMv / 16, QB = TNv / 16;          // elements per thread per 16-k step
  constexpr int BM = TMv / 32, BN = TNv / 32;          // MFMA blocks per wave
  auto &As = reinterpret_cast<GroupedShared<CPLX, TMv, TNv> *>(smem)->As;
  auto &Bs = reinterpret_cast<GroupedShared<CPLX, TMv, TNv> *>(smem)->Bs;

  const Seg seg = segs[tile.seg];
  const int i0 = tile.tm * TMv, j0 = tile.tn * TNv;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (w >> 1) * (TMv / 2), wn = (w & 1) * (TNv / 2);
  const int lr = lane & 15, lk = lane >> 4;

  v4d acc[BM][BN], acc_i[BM][BN], acc_s[BM][BN];
#pragma unroll
  for (int a = 0; a < BM; ++a)
#pragma unroll
    for (int b = 0; b < BN; ++b) {
      acc[a][b] = v4d{0.0, 0.0, 0.0, 0.0};
      acc_i[a][b] = v4d{0.0, 0.0, 0.0, 0.0};
      acc_s[a][b] = v4d{0.0, 0.0, 0.0, 0.0};
    }

  // ---- MFMAs on one staged step ----
  // Work outside the output block is skipped: 16 x 16 sub-blocks of the wave
  // that lie wholly beyond m or n, and halves of a chunk beyond its valid
  // extent `kv`, all wave-uniform.  The fragments of half a chunk are read
  // together, before its MFMAs: read one by one inside a guard, each MFMA
  // waited for its own LDS round trip (with the unguarded loads below, D = 2048
  // FP64 277 -> 249 us, D = 4096 complex128 1.17 -> 1.14 ms).
  bool mt_ok[BM], nt_ok[BN];
#pragma unroll
  for (int mt = 0; mt < BM; ++mt) mt_ok[mt] = i0 + wm + mt * 16 < seg.m;
#pragma unroll
  for (int nt = 0; nt < BN; ++nt) nt_ok[nt] = j0 + wn + nt * 16 < seg.n;
  const bool wave_on = mt_ok[0] && nt_ok[0];
  typedef double v2d __attribute__((ext_vector_type(2)));
  auto compute = [&](int kv) {
    if (!wave_on) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (8 * h >= kv) break;
      v2d a[BM], ai[BM];
      double b[2][BN], bi[2][BN];
#pragma unroll
      for (int mt = 0; mt < BM; ++mt) {
        a[mt] = *reinterpret_cast<const v2d *>(&As[0][wm + mt * 16 + lr][4 * lk + 2 * h]);
        if (CPLX) ai[mt] = *reinterpret_cast<const v2d *>(&As[P - 1][wm + mt * 16 + lr][4 * lk + 2 * h]);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int nt = 0; nt < BN; ++nt) {
          b[u][nt] = Bs[0][4 * lk + 2 * h + u][wn + nt * 16 + lr];
          if (CPLX) bi[u][nt] = Bs[P - 1][4 * lk + 2 * h + u][wn + nt * 16 + lr];
        }
#pragma unroll
      for (int mt = 0; mt < BM; ++mt) {
        if (mt > 0 && !mt_ok[mt]) continue;
#pragma unroll
        for (int nt = 0; nt < BN; ++nt) {
          if (nt > 0 && !nt_ok[nt]) continue;
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            acc[mt][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[mt][u], b[u][nt], acc[mt][nt], 0, 0, 0);
            if (CPLX) {
              // three real products per complex one (Gauss): acc = sum ar*br,
              // acc_i = sum ai*bi, acc_s = sum (ar + ai)*(br + bi); after the last
              // step re = acc - acc_i and im = acc_s - acc - acc_i
              acc_i[mt][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[mt][u], bi[u][nt], acc_i[mt][nt], 0, 0, 0);
              acc_s[mt][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[mt][u] + ai[mt][u], b[u][nt] + bi[u][nt],
                                                                   acc_s[mt][nt], 0, 0, 0);
            }
          }
        }
      }
    }
  };

  // ---- pipeline over this tile's steps of the (task, k-chunk) sequence ----
  // A step stages 16 k, never crossing a task.  Every load is issued without
  // a guard (guarded or in two versions of a step, the compiler waited for all
  // loads before issuing the last one): rows and columns past the block read its first ones (their
  // results are never stored), and contracted indices past the task read the
  // operand block's own elements and are staged as zero.
  const bool seg_plain = (seg.flags & (kSegAPlain | kSegBPlain)) == (kSegAPlain | kSegBPlain);
  const bool seg_affine = (seg.flags & (kSegAColAffine | kSegBRowAffine)) == (kSegAColAffine | kSegBRowAffine);
  raw_t<E, CPLX> pa[QA], pb[QB];
  int t = tile.t_begin, kk = tile.k_begin, left = tile.n_chunks;
  ExecTask et = exec[t];
  int kv = min(KC, et.k - kk);
  if (seg_affine) {
    // Output block whose every task reads A and B blocks that are affine in
    // k: A' element (r, p) at a_off + roff(r) + p * cs, B' element (p, c) at
    // b_off + p * rs + coff(c) (plain blocks: roff = r*k, cs = 1, rs = n,
    // coff = c).  Each thread keeps one pointer per element it loads, set
    // once per task (the row / column offsets decomposed there) and advanced
    // by 16 k per step.
    const int ap = tid & 15, ar0 = tid >> 4, apl = k_place(ap);
    const int bc = tid % TNv, bp0 = tid / TNv;
    constexpr int BPS = 256 / TNv;                     // B' rows between a thread's elements
    const E *aptr[QA], *bptr[QB], *a0 = A, *b0 = B;   // a0, b0: the task's blocks
    int64_t a_adv = 0, b_adv = 0;
    auto setup = [&](const ExecTask &e, int kk0) {
      const BlkGather &gA = ga[e.a_blk];
      const BlkGather &gB = gb[e.b_blk];
      const bool pa_ = seg_plain || gA.plain != 0, pb_ = seg_plain || gB.plain != 0;
      const int64_t cs = pa_ ? 1 : gA.cstep;
      const int64_t rs = pb_ ? seg.n : gB.rstep;
      a_adv = KC * cs * P;
      b_adv = KC * rs * P;
      a0 = A + e.a_off * P;
      b0 = B + e.b_off * P;
      PartSplit a_m{}, b_n{};
      if (!pa_) a_m = part_split<true>(gA, L.a_nr);
      if (!pb_) b_n = part_split<false>(gB, L.b_nc);
#pragma unroll
      for (int q = 0; q < QA; ++q) {
        const int r = i0 + ar0 + 16 * q < seg.m ? i0 + ar0 + 16 * q : 0;
        const int64_t roff = pa_ ? static_cast<int64_t>(r) * e.k : offset_of<true>(a_m, r);
        aptr[q] = a0 + (roff + (ap + kk0) * cs) * P;
      }
      const int c = j0 + bc < seg.n ? j0 + bc : 0;
      const int64_t coff = pb_ ? c : offset_of<false>(b_n, c);
#pragma unroll
      for (int q = 0; q < QB; ++q) bptr[q] = b0 + (static_cast<int64_t>(bp0 + BPS * q + kk0) * rs + coff) * P;
    };
    auto pfetch = [&](int kvalid) {
      if (kvalid < KC) {   // a task's last chunk: the pointers are set anew after it
#pragma unroll
        for (int q = 0; q < QA; ++q) aptr[q] = ap < kvalid ? aptr[q] : a0;
#pragma unroll
        for (int q = 0; q < QB; ++q) bptr[q] = bp0 + BPS * q < kvalid ? bptr[q] : b0;
      }
#pragma unroll
      for (int q = 0; q < QA; ++q) {
        pa[q] = ld_raw<E, CPLX>(aptr[q]);
        aptr[q] += a_adv;
      }
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        pb[q] = ld_raw<E, CPLX>(bptr[q]);
        bptr[q] += b_adv;
      }
    };
    auto pstage = [&](int kvalid) {
      if (kvalid < KC) {
#pragma unroll
        for (int q = 0; q < QA; ++q) zero_unless<E, CPLX>(pa[q], ap < kvalid);
#pragma unroll
        for (int q = 0; q < QB; ++q) zero_unless<E, CPLX>(pb[q], bp0 + BPS * q < kvalid);
      }
#pragma unroll
      for (int q = 0; q < QA; ++q) {
        As[0][ar0 + 16 * q][apl] = re_of(pa[q]);
        if (CPLX) As[P - 1][ar0 + 16 * q][apl] = im_of(pa[q]);
      }
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        Bs[0][k_place(bp0 + BPS * q)][bc] = re_of(pb[q]);
        if (CPLX) Bs[P - 1][k_place(bp0 + BPS * q)][bc] = im_of(pb[q]);
      }
    };
    setup(et, kk);
    pfetch(kv);
    pstage(kv);
    __syncthreads();
    for (;;) {
      --left;
      int kv2 = 0;
      if (left > 0) {
        kk += KC;
        if (kk >= et.k) {
          et = exec[++t];
          kk = 0;
          setup(et, 0);
        }
        kv2 = min(KC, et.k - kk);
        pfetch(kv2);
      }
      compute(kv);
      if (left == 0) break;
      __syncthreads();
      pstage(kv2);
      __syncthreads();
      kv = kv2;
    }
  } else {
    // Other blocks: offsets decomposed per element.  The thread mapping of a
    // chunk follows the block's innermost memory axis, chosen per task:
    //   A' k-contiguous -> p = tid & 15, rows (tid >> 4) + 16 q;
    //      otherwise    -> r = tid % TM, cols tid / TM + (256 / TM) q;
    //   B' n-contiguous -> c = tid % TN, rows tid / TN + (256 / TN) q;
    //      otherwise    -> p = tid & 15, cols (tid >> 4) + 16 q.
    bool akf = false, bnf = false, a_plain = false, b_plain = false;
    auto a_r = [&](int q) { return akf ? (tid >> 4) + 16 * q : tid % TMv; };
    auto a_p = [&](int q) { return akf ? tid & 15 : tid / TMv + (256 / TMv) * q; };
    auto b_c = [&](int q) { return bnf ? tid % TNv : (tid >> 4) + 16 * q; };
    auto b_p = [&](int q) { return bnf ? tid / TNv + (256 / TNv) * q : tid & 15; };
    int32_t a_row[QA], b_col[QB];
    PartSplit a_k{}, b_k{};
    auto task_rows = [&](const ExecTask &e) {
      const BlkGather &gA = ga[e.a_blk];
      const BlkGather &gB = gb[e.b_blk];
      a_plain = gA.plain != 0;
      b_plain = gB.plain != 0;
      akf = a_plain || gA.fastcol != 0;
      bnf = b_plain || gB.fastcol != 0;
      a_k = part_split<false>(gA, L.a_nc);
      b_k = part_split<true>(gB, L.b_nr);
      const PartSplit a_m = part_split<true>(gA, L.a_nr);
      const PartSplit b_n = part_split<false>(gB, L.b_nc);
#pragma unroll
      for (int q = 0; q < QA; ++q) {
        const int r = i0 + a_r(q) < seg.m ? i0 + a_r(q) : 0;
        a_row[q] = a_plain ? r * e.k : offset_of<true>(a_m, r);
      }
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        const int c = j0 + b_c(q) < seg.n ? j0 + b_c(q) : 0;
        b_col[q] = b_plain ? c : offset_of<false>(b_n, c);
      }
    };
    auto fetch = [&](const ExecTask &e, int k0, int kvalid) {
#pragma unroll
      for (int q = 0; q < QA; ++q) {
        const int pk = k0 + (a_p(q) < kvalid ? a_p(q) : 0);
        const int32_t col = a_plain ? pk : offset_of<false>(a_k, pk);
        pa[q] = ld_raw<E, CPLX>(A + (e.a_off + a_row[q] + col) * P);
      }
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        const int pk = k0 + (b_p(q) < kvalid ? b_p(q) : 0);
        const int32_t row = b_plain ? pk * seg.n : offset_of<true>(b_k, pk);
        pb[q] = ld_raw<E, CPLX>(B + (e.b_off + row + b_col[q]) * P);
      }
    };
    auto stage = [&](int kvalid) {
      if (kvalid < KC) {
#pragma unroll
        for (int q = 0; q < QA; ++q) zero_unless<E, CPLX>(pa[q], a_p(q) < kvalid);
#pragma unroll
        for (int q = 0; q < QB; ++q) zero_unless<E, CPLX>(pb[q], b_p(q) < kvalid);
      }
#pragma unroll
      for (int q = 0; q < QA; ++q) {
        As[0][a_r(q)][k_place(a_p(q))] = re_of(pa[q]);
        if (CPLX) As[P - 1][a_r(q)][k_place(a_p(q))] = im_of(pa[q]);
      }
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        Bs[0][k_place(b_p(q))][b_c(q)] = re_of(pb[q]);
        if (CPLX) Bs[P - 1][k_place(b_p(q))][b_c(q)] = im_of(pb[q]);
      }
    };
    task_rows(et);
    fetch(et, kk, kv);
    stage(kv);
    __syncthreads();
    for (;;) {
      --left;
      int kv2 = 0;
      if (left > 0) {
        kk += KC;
        if (kk >= et.k) {
          et = exec[++t];
          kk = 0;
          task_rows(et);
        }
        kv2 = min(KC, et.k - kk);
        fetch(et, kk, kv2);
      }
      compute(kv);
      if (left == 0) break;
      __syncthreads();
      stage(kv2);
      __syncthreads();
      kv = kv2;
    }
  }

  // ---- complex: the real and imaginary parts from the three product sums ----
  if (CPLX) {
#pragma unroll
    for (int mt = 0; mt < BM; ++mt)
#pragma unroll
      for (int nt = 0; nt < BN; ++nt) {
        const v4d p1 = acc[mt][nt], p2 = acc_i[mt][nt];
        acc[mt][nt] = p1 - p2;
        acc_i[mt][nt] = acc_s[mt][nt] - p1 - p2;
      }
  }

  // ---- a k-slice stores its unscaled partial sum, row-major over the tile ----
  if (tile.part >= 0) {
    double *pp = part + static_cast<int64_t>(tile.part) * (TMv * TNv * P);
#pragma unroll
    for (int mt = 0; mt < BM; ++mt)
#pragma unroll
      for (int nt = 0; nt < BN; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int e = (wm + 16 * mt + 4 * v + lk) * TNv + wn + 16 * nt + lr;
          pp[e] = acc[mt][nt][v];
          if (CPLX) pp[TMv * TNv + e] = acc_i[mt][nt][v];
        }
    return;
  }

  // ---- epilogue: C = alpha * acc + beta * C (C untouched when beta == 0) ----
  // f64 16x16x4 output: row 4*reg + lane/16
  tile_epilogue<CPLX, BM, BN, E>(seg, i0 + wm + lk, j0 + wn + lr, acc, acc_i, C, alpha_r, alpha_i, beta_r, beta_i);
}

// Narrow outputs (n <= 16): 32 x 16 tiles of two MFMA blocks of 16 x 16.  KW = 4: a
// workgroup takes one tile or k-slice of it, its four waves every fourth
// 16-k chunk of the tile's (task, chunk) sequence, and they meet in LDS at the
// end (sums in wave order).  KW = 1: a workgroup takes four tiles, a wave each,
// which walks all of its tile's chunks.  The operand fragments are loaded from
// global memory straight into the registers the MFMA reads (lane lr = lane % 16
// holds A' row / B' column lr, lk = lane / 16 the contracted index), so no wave
// waits for another inside the loop, and the loads of one stage are issued before
// the MFMAs of the previous one (two register sets).
//   What bounds it is latency: with KW = 4 of few tiles, each a long chain of
// chunks, which a kernel with one thread per row and an LDS chunk of B' per step
// walked alone, about 1 us per 16 k: a complex64 contraction onto n <= 16 outputs
// 143 -> 27 us, the n <= 16 tiles of a lognormal FP64 matvec 46 -> 15 us per
// contraction.  With KW = 1 of many tiles of few chunks: the chain of a tile's
// records, its loads and its stores, against the waves in flight (complex: two k-steps
// a stage instead of four for them; n = 8, k = 16, m = 10^6, complex64: 150 us with KW = 4, 77
// with four, 69 with two; one thread per row 82).  The same unstaged form for n > 16
// is slower than the LDS tiles (D = 4096 complex128 matvec 1.23 -> 1.41 ms): there the
// fragments' uncoalesced lines bound it, so it stays with these classes.
//   Full stages of the types of at most 8 bytes per element give lane (lr, lk)
// the KS consecutive contracted indices KS lk .. KS lk + KS - 1, so that an
// operand contiguous in k is read in 16-byte pieces; complex128 and a task's
// last partial stage use 4 s + lk.  The order of the contracted indices is
// free as long as both operands follow it.
//   Rows and columns past the block read the block's first row or column and
// their results are not stored; contracted indices past the task count zero
// on both sides.
constexpr int kNarrowM = 32, kNarrowN = 16, kNarrowWaves = 4;

template <bool CPLX>
struct NarrowShared {
  double acc[kNarrowWaves][CPLX ? 2 : 1][2][4][64];
};

// KS consecutive elements of an operand contiguous in k: 16-byte loads with
// the element's alignment only.
template <typename E, bool CPLX, int KS>
__device__ __forceinline__ void ld_run(const E *p, raw_t<E, CPLX> (&x)[KS]) {
  static_assert(sizeof(raw_t<E, CPLX>) <= 8, "runs are for elements of at most 8 bytes");
  typedef E vec __attribute__((ext_vector_type(16 / sizeof(E)), aligned(sizeof(E))));
  constexpr int PER = 16 / sizeof(raw_t<E, CPLX>);   // elements per load
  static_assert(KS % PER == 0, "whole 16-byte pieces");
#pragma unroll
  for (int i = 0; i < KS / PER; ++i) {
    const vec v = reinterpret_cast<const vec *>(p)[i];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      if constexpr (CPLX) x[i * PER + j] = raw_t<E, CPLX>{v[2 * j], v[2 * j + 1]};
      else x[i * PER + j] = v[j];
    }
  }
}

template <bool CPLX, int KW, typename E>
__device__ __forceinline__ void narrow_tile(
    char *smem, const Tile tile, const Seg *__restrict__ segs, const ExecTask *__restrict__ exec,
    const BlkGather *__restrict__ ga, const BlkGather *__restrict__ gb, const GatherLayout &L,
    const E *__restrict__ A, const E *__restrict__ B, E *__restrict__ C, double *__restrict__ part,
    double alpha_r, double alpha_i, double beta_r, double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  constexpr int BM = kNarrowM / 16;
  constexpr int kTileRows = kNarrowM * (kNarrowWaves / KW);   // of the workgroup
  // k-steps of 4 per stage: their registers bound k_all_classes (KW = 4) and the waves in flight (KW = 1)
  constexpr int KS = sizeof(E) == 8 || (CPLX && KW == 1) ? 2 : 4;
  constexpr int SK = 4 * KS;
  constexpr bool kLaneRuns = sizeof(E) * P <= 8;
  using R = raw_t<E, CPLX>;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const Seg seg = segs[tile.seg];
  const int wk = KW > 1 ? w : 0;                              // the wave's place in its tile's chunks
  const int r0 = KW > 1 ? 0 : kNarrowM * w;                   // its rows' place in the workgroup's
  const int i0 = tile.tm * kTileRows + r0;
  if (KW == 1 && i0 >= seg.m) return;
  const bool m1_ok = i0 + 16 < seg.m;
  v4d acc[P][BM];
#pragma unroll
  for (int q = 0; q < P; ++q)
#pragma unroll
    for (int mt = 0; mt < BM; ++mt) acc[q][mt] = v4d{0.0, 0.0, 0.0, 0.0};
  R a[2][BM][KS], b[2][KS];

  // position: task t (k extent tk), contracted index kk, chunks left
  int t = tile.t_begin, kk = tile.k_begin, left = tile.n_chunks - wk;
  int tk = 0;
  // moves n chunks forward from chunk start kk (which may equal or pass tk)
  auto skip = [&](int n) {
    for (;;) {
      if (kk >= tk) {
        ++t;
        tk = exec[t].k;
        kk = 0;
      }
      if (n == 0) break;
      const int here = chunks_from(kk, tk);
      if (n < here) {
        kk += KC * n;
        break;
      }
      n -= here;
      kk = tk;
    }
  };

  // per task: element pointers of this lane's rows and column at k = 0, and
  // how an index k moves them
  const E *ap[BM], *bp = nullptr;
  PartSplit a_k{}, b_k{};
  bool a_aff = false, b_aff = false;
  int cs = 1, rs = 1, cur = -1;
  auto setup = [&]() {
    cur = t;
    const ExecTask et = exec[t];
    const BlkGather &gA = ga[et.a_blk];
    const BlkGather &gB = gb[et.b_blk];
    const bool a_plain = (seg.flags & kSegAPlain) || gA.plain != 0;
    const bool b_plain = (seg.flags & kSegBPlain) || gB.plain != 0;
    a_aff = (seg.flags & kSegAColAffine) || a_plain || gA.caff != 0;
    b_aff = (seg.flags & kSegBRowAffine) || b_plain || gB.raff != 0;
    cs = a_plain ? 1 : gA.cstep;
    rs = b_plain ? seg.n : gB.rstep;
    PartSplit a_m{}, b_n{};
    if (!a_plain) a_m = part_split<true>(gA, L.a_nr);
    if (!b_plain) b_n = part_split<false>(gB, L.b_nc);
    if (!a_aff) a_k = part_split<false>(gA, L.a_nc);
    if (!b_aff) b_k = part_split<true>(gB, L.b_nr);
#pragma unroll
    for (int mt = 0; mt < BM; ++mt) {
      int r = i0 + 16 * mt + lr;
      r = r < seg.m ? r : 0;
      ap[mt] = A + (et.a_off + (a_plain ? static_cast<int64_t>(r) * et.k : offset_of<true>(a_m, r))) * P;
    }
    const int c = lr < seg.n ? lr : 0;
    bp = B + (et.b_off + (b_plain ? c : offset_of<false>(b_n, c))) * P;
  };
  auto a_off = [&](int k) -> int64_t { return a_aff ? static_cast<int64_t>(k) * cs : offset_of<false>(a_k, k); };
  auto b_off = [&](int k) -> int64_t { return b_aff ? static_cast<int64_t>(k) * rs : offset_of<true>(b_k, k); };
  // the stage at (t, kk) into register set `s`; returns its valid extent
  auto load = [&](int s) {
    if (t != cur) setup();
    const int kv = tk - kk < SK ? tk - kk : SK;
    if (kv == SK) {
      bool a_run = false, b_run = false;
      if constexpr (kLaneRuns) {
        a_run = a_aff && cs == 1;
        b_run = b_aff && rs == 1;
        if (a_run) {
          ld_run<E, CPLX, KS>(ap[0] + run_offset(kk + KS * lk, P), a[s][0]);
          if (m1_ok) ld_run<E, CPLX, KS>(ap[1] + run_offset(kk + KS * lk, P), a[s][1]);
        }
        if (b_run) ld_run<E, CPLX, KS>(bp + run_offset(kk + KS * lk, P), b[s]);
      }
      if (!a_run) {
#pragma unroll
        for (int q = 0; q < KS; ++q) {
          const int64_t off = a_off(kk + (kLaneRuns ? KS * lk + q : 4 * q + lk)) * P;
          a[s][0][q] = ld_raw<E, CPLX>(ap[0] + off);
          if (m1_ok) a[s][1][q] = ld_raw<E, CPLX>(ap[1] + off);
        }
      }
      if (!b_run) {
#pragma unroll
        for (int q = 0; q < KS; ++q)
          b[s][q] = ld_raw<E, CPLX>(bp + b_off(kk + (kLaneRuns ? KS * lk + q : 4 * q + lk)) * P);
      }
    } else {
      // a task's last stage: k = kk + 4 q + lk, the steps beyond it skipped
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        if (4 * q >= kv) continue;
        const bool ok = 4 * q + lk < kv;
        const int k = ok ? kk + 4 * q + lk : kk;
        const int64_t ao = a_off(k) * P;
        const R x = ld_raw<E, CPLX>(ap[0] + ao), z = ld_raw<E, CPLX>(bp + b_off(k) * P);
        a[s][0][q] = ok ? x : R{};
        b[s][q] = ok ? z : R{};
        if (m1_ok) {
          const R y = ld_raw<E, CPLX>(ap[1] + ao);
          a[s][1][q] = ok ? y : R{};
        }
      }
    }
    return kv;
  };
  auto compute = [&](int s, int kv) {
#pragma unroll
    for (int q = 0; q < KS; ++q) {
      if (kv < SK && 4 * q >= kv) continue;
      const double br = re_of(b[s][q]), bi = im_of(b[s][q]);
#pragma unroll
      for (int mt = 0; mt < BM; ++mt) {
        if (mt == 1 && !m1_ok) continue;
        const double ar = re_of(a[s][mt][q]);
        v4d &x = acc[0][mt];
        x = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, x, 0, 0, 0);
        if constexpr (CPLX) {
          // four real products: this class is not bound by them
          const double ai = im_of(a[s][mt][q]);
          v4d &y = acc[P - 1][mt];
          x = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, bi, x, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, y, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, y, 0, 0, 0);
        }
      }
    }
  };
  // past the stage of extent kv; false when this wave's chunks are done
  auto advance = [&](int kv) {
    kk += kv;
    if (kk < tk && (kk & (KC - 1)) != 0) return true;   // inside a chunk
    left -= KW;
    if (left <= 0) return false;
    skip(KW - 1);
    return true;
  };
  if (left > 0) {
    tk = exec[t].k;
    skip(wk);
    int kv0 = load(0);
    for (;;) {
      bool more = advance(kv0);
      int kv1 = 0;
      if (more) kv1 = load(1);
      compute(0, kv0);
      if (!more) break;
      more = advance(kv1);
      if (more) kv0 = load(0);
      compute(1, kv1);
      if (!more) break;
    }
  }

  if constexpr (KW == 1) {
    // element v of a lane is row 4 v + lk of its MFMA block; a k-slice stores its
    // unscaled partial sum, row-major over the workgroup's rows
    double *pp = tile.part >= 0 ? part + static_cast<int64_t>(tile.part) * (kTileRows * kNarrowN * P) : nullptr;
    const bool use_beta = pp == nullptr && (beta_r != 0.0 || beta_i != 0.0);
    R old[BM][4];
#pragma unroll
    for (int mt = 0; mt < BM; ++mt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        old[mt][v] = R{};
        if (use_beta) {
          const int row = i0 + 16 * mt + 4 * v + lk;
          const bool ok = row < seg.m && lr < seg.n;
          old[mt][v] = ld_raw<E, CPLX>(C + P * (seg.c_off + (ok ? static_cast<int64_t>(row) * seg.n + lr : 0)));
        }
      }
#pragma unroll
    for (int mt = 0; mt < BM; ++mt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int lrow = 16 * mt + 4 * v + lk;
        const double xr = acc[0][mt][v], xi = CPLX ? acc[P - 1][mt][v] : 0.0;
        if (pp != nullptr) {
          pp[(r0 + lrow) * kNarrowN + lr] = xr;
          if (CPLX) pp[kTileRows * kNarrowN + (r0 + lrow) * kNarrowN + lr] = xi;
        } else if (i0 + lrow < seg.m && lr < seg.n) {
          st_scaled<E, CPLX>(C + P * (seg.c_off + static_cast<int64_t>(i0 + lrow) * seg.n + lr), xr, xi, old[mt][v],
                             use_beta, alpha_r, alpha_i, beta_r, beta_i);
        }
      }
    return;
  }

  // wave w takes the accumulator element v = w of every lane, from all waves
  auto &sAcc = reinterpret_cast<NarrowShared<CPLX> *>(smem)->acc;
#pragma unroll
  for (int q = 0; q < P; ++q)
#pragma unroll
    for (int mt = 0; mt < BM; ++mt)
#pragma unroll
      for (int v = 0; v < 4; ++v) sAcc[w][q][mt][v][lane] = acc[q][mt][v];
  __syncthreads();
  double *pp = tile.part >= 0 ? part + static_cast<int64_t>(tile.part) * (kNarrowM * kNarrowN * P) : nullptr;
  const bool use_beta = pp == nullptr && (beta_r != 0.0 || beta_i != 0.0);
  double xr[BM], xi[BM];
  R old[BM];
#pragma unroll
  for (int mt = 0; mt < BM; ++mt) {
    xr[mt] = 0.0;
    xi[mt] = 0.0;
#pragma unroll
    for (int g = 0; g < KW; ++g) {
      xr[mt] += sAcc[g][0][mt][w][lane];
      if (CPLX) xi[mt] += sAcc[g][P - 1][mt][w][lane];
    }
    old[mt] = R{};
    if (use_beta) {
      const int row = i0 + 16 * mt + 4 * w + lk;
      const bool ok = row < seg.m && lr < seg.n;
      old[mt] = ld_raw<E, CPLX>(C + P * (seg.c_off + (ok ? static_cast<int64_t>(row) * seg.n + lr : 0)));
    }
  }
#pragma unroll
  for (int mt = 0; mt < BM; ++mt) {
    const int lrow = 16 * mt + 4 * w + lk;
    if (pp != nullptr) {
      // a k-slice stores its unscaled partial sum, row-major over the tile
      pp[lrow * kNarrowN + lr] = xr[mt];
      if (CPLX) pp[kNarrowM * kNarrowN + lrow * kNarrowN + lr] = xi[mt];
    } else if (i0 + lrow < seg.m && lr < seg.n) {
      st_scaled<E, CPLX>(C + P * (seg.c_off + static_cast<int64_t>(i0 + lrow) * seg.n + lr), xr[mt], xi[mt], old[mt],
                         use_beta, alpha_r, alpha_i, beta_r, beta_i);
    }
  }
}

// Sum of the k-slices of one output tile, in slice order, then the usual
// epilogue: element e of the tile (row-major) in thread e % 256.
template <bool CPLX, int TMv, int TNv, typename E>
__device__ __forceinline__ void reduce_slices(const ReduceItem it, const Seg &seg, const double *__restrict__ part,
                                              E *__restrict__ C, double alpha_r, double alpha_i, double beta_r,
                                              double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  constexpr int NE = TMv * TNv / 256;
  const int tid = threadIdx.x;
  double sr[NE], si[NE];
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    sr[u] = 0.0;
    si[u] = 0.0;
  }
  // slices outer, elements inner: every slice's loads are independent
  for (int s = 0; s < it.n_parts; ++s) {
    const double *pp = part + static_cast<int64_t>(it.part0 + s) * (TMv * TNv * P);
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      sr[u] += pp[tid + 256 * u];
      if (CPLX) si[u] += pp[TMv * TNv + tid + 256 * u];
    }
  }
  const bool use_beta = beta_r != 0.0 || beta_i != 0.0;
  raw_t<E, CPLX> old[NE];
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = tid + 256 * u, row = it.tm * TMv + e / TNv, col = it.tn * TNv + e % TNv;
    const bool ok = row < seg.m && col < seg.n;
    old[u] = raw_t<E, CPLX>{};
    if (use_beta) old[u] = ld_raw<E, CPLX>(C + P * (seg.c_off + (ok ? static_cast<int64_t>(row) * seg.n + col : 0)));
  }
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = tid + 256 * u, row = it.tm * TMv + e / TNv, col = it.tn * TNv + e % TNv;
    if (row < seg.m && col < seg.n)
      st_scaled<E, CPLX>(C + P * (seg.c_off + static_cast<int64_t>(row) * seg.n + col), sr[u], si[u], old[u], use_beta,
                         alpha_r, alpha_i, beta_r, beta_i);
  }
}

// Row-streaming kernel for narrow outputs (n <= NMAX): one thread per output
// row, RPT rows per thread (rows tid, tid + 256, ...).  A' is read straight
// from global memory -- consecutive rows are consecutive threads, so the
// loads are contiguous whenever A's innermost axis is a saved one, and with
// RPT independent rows each thread keeps several loads in flight.  The
// 16 x n chunk of B' is staged once per workgroup in LDS and every thread
// accumulates its n outputs with FP64 FMAs.  Bound by reading A and writing
// C once.
constexpr int RK = 16;            // k per stage
// A loads in flight per thread.  A row of 16 contiguous k is one memory line, which
// a step touches once per group: eight loads at a time instead of sixteen cost
// up to half of the time (n = 4, k = 16, m = 10^6, FP64: 141 -> 230 us, with the vector
// loads that k_row_class avoids).
constexpr int kRowsLoadGroup = 16;

template <bool CPLX, int NMAX, int RPT, typename E>
__device__ __forceinline__ void rows_epilogue(const Seg &seg, int r0, int tid, const double (&acc)[RPT][NMAX],
                                              const double (&acc_i)[RPT][NMAX], E *__restrict__ C,
                                              double alpha_r, double alpha_i, double beta_r, double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  const int n = seg.n;
  // beta == 0 and beta != 0 as separate code, as in tile_epilogue
  auto store_all = [&](auto with_beta, const raw_t<E, CPLX>(&old)[RPT][NMAX]) {
    constexpr bool WB = decltype(with_beta)::value;
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      const int row = r0 + tid + 256 * q;
      if (row >= seg.m) continue;
      const int64_t base = seg.c_off + static_cast<int64_t>(row) * n;
#pragma unroll
      for (int j = 0; j < NMAX; ++j) {
        if (j < n) {
          st_scaled<E, CPLX>(C + P * (base + j), acc[q][j], CPLX ? acc_i[q][j] : 0.0, old[q][j], WB,
                             alpha_r, alpha_i, beta_r, beta_i);
        }
      }
    }
  };
  if (beta_r != 0.0 || beta_i != 0.0) {
    raw_t<E, CPLX> old[RPT][NMAX];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      const int row = r0 + tid + 256 * q;
#pragma unroll
      for (int j = 0; j < NMAX; ++j) {
        const bool ok = row < seg.m && j < n;
        old[q][j] = ld_raw<E, CPLX>(C + P * (seg.c_off + (ok ? static_cast<int64_t>(row) * n + j : 0)));
      }
    }
    store_all(std::true_type{}, old);
  } else {
    const raw_t<E, CPLX> none[RPT][NMAX] = {};
    store_all(std::false_type{}, none);
  }
}

template <bool CPLX, int NMAX>
struct RowsShared {
  double Bs[CPLX ? 2 : 1][RK][NMAX];
  int32_t acol[RK], brow[RK], bcol[NMAX];
};
template <bool CPLX, int NMAX, int RPT, typename E>
__device__ __forceinline__ void rows_tile(
    char *smem, const Tile tile, const Seg *__restrict__ segs, const ExecTask *__restrict__ exec,
    const BlkGather *__restrict__ ga, const BlkGather *__restrict__ gb, const GatherLayout &L,
    const E *__restrict__ A, const E *__restrict__ B, E *__restrict__ C, double *__restrict__ part,
    double alpha_r, double alpha_i, double beta_r, double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  static_assert(RK * NMAX <= 256, "one B' element per thread");
  static_assert(RK == kKChunk, "row kernel steps are the plan's k-chunks");
  auto &Bs = reinterpret_cast<RowsShared<CPLX, NMAX> *>(smem)->Bs;
  auto &s_acol = reinterpret_cast<RowsShared<CPLX, NMAX> *>(smem)->acol;
  auto &s_brow = reinterpret_cast<RowsShared<CPLX, NMAX> *>(smem)->brow;
  auto &s_bcol = reinterpret_cast<RowsShared<CPLX, NMAX> *>(smem)->bcol;

  const Seg seg = segs[tile.seg];
  const int tid = threadIdx.x;
  const int r0 = tile.tm * (256 * RPT);
  const int n = seg.n;

  double acc[RPT][NMAX], acc_i[RPT][NMAX];
#pragma unroll
  for (int q = 0; q < RPT; ++q)
#pragma unroll
    for (int j = 0; j < NMAX; ++j) {
      acc[q][j] = 0.0;
      acc_i[q][j] = 0.0;
    }

  // this tile's steps of the (task, k-chunk) sequence
  int t = tile.t_begin, kk = tile.k_begin;
  ExecTask et{};
  bool a_plain = false, b_plain = false;
  int32_t roff[RPT];
  int cur_task = -1;
  for (int step = 0; step < tile.n_chunks; ++step) {
    if (t != cur_task) {
      cur_task = t;
      et = exec[t];
      const BlkGather &gA = ga[et.a_blk];
      const BlkGather &gB = gb[et.b_blk];
      a_plain = gA.plain != 0;
      b_plain = gB.plain != 0;
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        const int row = r0 + tid + 256 * q;
        roff[q] = (row < seg.m) ? (a_plain ? row * et.k : split_offset(row, gA.rdim, gA.rstr, gA.rmag, gA.rsh, L.a_nr)) : -1;
      }
      __syncthreads();
      if (tid < NMAX)
        s_bcol[tid] = (tid < n) ? (b_plain ? tid : split_offset(tid, gB.cdim, gB.cstr, gB.cmag, gB.csh, L.b_nc)) : -1;
    }
    const BlkGather &gA = ga[et.a_blk];
    const BlkGather &gB = gb[et.b_blk];
    if (tid < RK) {
      const int p = kk + tid;
      s_acol[tid] = (p < et.k) ? (a_plain ? p : split_offset(p, gA.cdim, gA.cstr, gA.cmag, gA.csh, L.a_nc)) : -1;
    } else if (tid >= 64 && tid < 64 + RK) {
      const int p = kk + tid - 64;
      s_brow[tid - 64] = (p < et.k) ? (b_plain ? p * n : split_offset(p, gB.rdim, gB.rstr, gB.rmag, gB.rsh, L.b_nr)) : -1;
    }
    __syncthreads();
    if (tid < RK * NMAX) {
      const int p = tid / NMAX, j = tid % NMAX;
      const int32_t ro = s_brow[p], co = s_bcol[j];
      const bool ok = (ro >= 0) && (co >= 0);
      const int64_t e = et.b_off + ro + co;
      const double2 v = ok ? ld_elem<E, CPLX>(B + e * P) : double2{0.0, 0.0};
      Bs[0][p][j] = v.x;
      if (CPLX) Bs[P - 1][p][j] = v.y;
    }
    __syncthreads();
    const int kc = min(RK, et.k - kk);
    // The A loads of G consecutive k steps go out together (G * RPT = 16 per
    // thread); a step beyond the chunk or a row beyond the block loads the
    // block's first element and counts zero.
#pragma unroll
    for (int p0 = 0; p0 < RK; p0 += kRowsLoadGroup / RPT) {
      constexpr int G = kRowsLoadGroup / RPT;
      if (p0 < kc) {
        double av[G][RPT], av_i[G][RPT];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int32_t co = s_acol[p0 + g];
#pragma unroll
          for (int q = 0; q < RPT; ++q) {
            const bool ok = roff[q] >= 0 && co >= 0;
            const double2 v = ld_elem<E, CPLX>(A + (ok ? et.a_off + roff[q] + co : et.a_off) * P);
            av[g][q] = ok ? v.x : 0.0;
            av_i[g][q] = ok ? v.y : 0.0;
          }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (p0 + g >= kc) continue;
          const int p = p0 + g;
#pragma unroll
          for (int j = 0; j < NMAX; ++j) {
            if (j < n) {
              const double b = Bs[0][p][j];
              const double b_im = Bs[P - 1][p][j];
#pragma unroll
              for (int q = 0; q < RPT; ++q) {
                if (CPLX) {
                  acc[q][j] = fma(av[g][q], b, acc[q][j]);
                  acc[q][j] = fma(-av_i[g][q], b_im, acc[q][j]);
                  acc_i[q][j] = fma(av[g][q], b_im, acc_i[q][j]);
                  acc_i[q][j] = fma(av_i[g][q], b, acc_i[q][j]);
                } else {
                  acc[q][j] = fma(av[g][q], b, acc[q][j]);
                }
              }
            }
          }
        }
      }
    }
    __syncthreads();
    kk += RK;
    if (kk >= et.k) {
      ++t;
      kk = 0;
    }
  }

  if (tile.part >= 0) {
    // k-slice: unscaled partial sums in the thread's own order
    double *pp = part + static_cast<int64_t>(tile.part) * (256 * RPT * NMAX * P);
#pragma unroll
    for (int q = 0; q < RPT; ++q)
#pragma unroll
      for (int j = 0; j < NMAX; ++j) {
        const int e = (q * NMAX + j) * 256 + tid;
        pp[e] = acc[q][j];
        if (CPLX) pp[256 * RPT * NMAX + e] = acc_i[q][j];
      }
    return;
  }
  rows_epilogue<CPLX, NMAX, RPT, E>(seg, r0, tid, acc, acc_i, C, alpha_r, alpha_i, beta_r, beta_i);
}

// Sum of the k-slices of one row tile, in slice order, then the epilogue.
template <bool CPLX, int NMAX, int RPT, typename E>
__device__ __forceinline__ void reduce_rows(const ReduceItem it, const Seg &seg, const double *__restrict__ part,
                                            E *__restrict__ C, double alpha_r, double alpha_i, double beta_r,
                                            double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  constexpr int SZ = 256 * RPT * NMAX * P;
  const int tid = threadIdx.x;
  double acc[RPT][NMAX], acc_i[RPT][NMAX];
#pragma unroll
  for (int q = 0; q < RPT; ++q)
#pragma unroll
    for (int j = 0; j < NMAX; ++j) {
      acc[q][j] = 0.0;
      acc_i[q][j] = 0.0;
    }
  // Each slice's slab holds the full RPT x NMAX layout, so every load is in
  // bounds; columns j >= n are loaded and dropped, which keeps the loads of a
  // slice in flight together.
  for (int s = 0; s < it.n_parts; ++s) {
    const double *pp = part + static_cast<int64_t>(it.part0 + s) * SZ;
#pragma unroll
    for (int q = 0; q < RPT; ++q)
#pragma unroll
      for (int j = 0; j < NMAX; ++j) {
        const int e = (q * NMAX + j) * 256 + tid;
        const bool ok = j < seg.n;
        const double x = pp[e];
        acc[q][j] += ok ? x : 0.0;
        if (CPLX) {
          const double xi = pp[256 * RPT * NMAX + e];
          acc_i[q][j] += ok ? xi : 0.0;
        }
      }
  }
  rows_epilogue<CPLX, NMAX, RPT, E>(seg, it.tm * (256 * RPT), tid, acc, acc_i, C, alpha_r, alpha_i, beta_r, beta_i);
}

// Row panels (PanelTile): one 512-row tile of a panel per workgroup, 2 rows
// per thread.  While each thread loads the A' elements of its rows in every
// column of the panel, the panel's terms (their B' elements, one thread
// each) and output columns are staged in LDS; then each output column is
// summed from registers in the row kernel's order and stored with its alpha
// / beta epilogue.  Replaces, for these blocks, the per-task loop of
// global_operations.h:919-978 (one BLAS call per task).
template <bool CPLX>
struct PanelShared {
  double br[kPanelMaxTerms], bi[kPanelMaxTerms];
  double pa[2][kPanelRows], pai[CPLX ? 2 : 1][kPanelRows];
  int64_t ocoff[kPanelMaxOuts];
  int32_t on[kPanelMaxOuts], ot0[kPanelMaxOuts], omask[kPanelMaxOuts];
};
template <bool CPLX, bool STREAM, typename E>
__device__ __forceinline__ void panel_tile(char *smem, const PanelTile &pt, const PanelOut *__restrict__ outs,
                                           const PanelTerm *__restrict__ terms, const Seg *__restrict__ segs,
                                           const E *__restrict__ A, const E *__restrict__ B, E *__restrict__ C,
                                           double alpha_r, double alpha_i, double beta_r, double beta_i) {
  constexpr int P = CPLX ? 2 : 1;
  constexpr int RPT = kPanelRpt;
  static_assert(kPanelRows == 512 && RPT == 2, "pair staging: 4 loads per thread");
  auto *sh = reinterpret_cast<PanelShared<CPLX> *>(smem);
  auto &s_br = sh->br, &s_bi = sh->bi;
  auto &s_pa = sh->pa;
  auto &s_pai = sh->pai;
  auto &s_ocoff = sh->ocoff;
  auto &s_on = sh->on, &s_ot0 = sh->ot0, &s_omask = sh->omask;
  static_assert(kPanelMaxTerms <= 128 && kPanelMaxOuts <= 128, "one staging thread per term and per output");

  const int tid = threadIdx.x;
  const int n_cols = pt.n_cols, n_outs = pt.n_outs, n_terms = pt.n_terms;

  // row offsets in every column: the row's digits over rdim (axes past the
  // saved ones have extent 1 and stride 0), dotted with each column's
  // strides.  Rows past the block read its first row (in bounds); their
  // sums are never stored, and the columns past n_cols are never read.
  int32_t roff[kPanelCols][RPT];
  bool valid[RPT];
#pragma unroll
  for (int q = 0; q < RPT; ++q) {
    const int row = pt.r0 + tid + 256 * q;
    valid[q] = row < pt.m;
    int32_t x = valid[q] ? row : 0;
#pragma unroll
    for (int c = 0; c < kPanelCols; ++c) roff[c][q] = 0;
#pragma unroll
    for (int l = kPanelRowAxes - 1; l >= 0; --l) {
      const int32_t qd = static_cast<int32_t>((static_cast<uint64_t>(x) * pt.rmag[l]) >> pt.rsh[l]);
      const int32_t d = x - qd * pt.rdim[l];
      x = qd;
#pragma unroll
      for (int c = 0; c < kPanelCols; ++c) roff[c][q] += d * pt.cstr[c][l];
    }
  }
  // every A' load is issued before anything waits on memory; each A'
  // element is read once, so when the panels' data exceed the last-level
  // cache (STREAM) the loads carry the non-temporal hint.  A pair
  // of columns that are adjacent elements of one A block (pt.pair1 - 1 and
  // pt.pair1) is loaded as (row, column) = (e / 2, e % 2) over the lanes, so
  // that one instruction reads both columns of 32 consecutive rows, and
  // reaches its rows' threads through LDS.
  const int pc = pt.pair1 - 1;   // first column of the pair, or -1
  double av[kPanelCols][RPT], av_i[kPanelCols][RPT];
  if (pc >= 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int rl = (tid >> 1) + 128 * j, cc = tid & 1;
      const int row = pt.r0 + rl;
      int32_t x = row < pt.m ? row : 0, off = 0;
#pragma unroll
      for (int l = kPanelRowAxes - 1; l >= 0; --l) {
        const int32_t qd = static_cast<int32_t>((static_cast<uint64_t>(x) * pt.rmag[l]) >> pt.rsh[l]);
        off += (x - qd * pt.rdim[l]) * pt.cstr[pc][l];
        x = qd;
      }
      const E *ap = A + (pt.cbase[pc] + off + cc) * P;
      const double2 v = STREAM ? ld_elem_stream<E, CPLX>(ap) : ld_elem<E, CPLX>(ap);
      s_pa[cc][rl] = v.x;
      if (CPLX) s_pai[CPLX ? cc : 0][rl] = v.y;
    }
  }
#pragma unroll
  for (int c = 0; c < kPanelCols; ++c)
    if (c < n_cols && (pc < 0 || (c != pc && c != pc + 1))) {
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        const E *ap = A + (pt.cbase[c] + roff[c][q]) * P;
        const double2 v = STREAM ? ld_elem_stream<E, CPLX>(ap) : ld_elem<E, CPLX>(ap);
        av[c][q] = v.x;
        av_i[c][q] = v.y;
      }
    }
  // stage the terms (B' elements) and the output columns
  if (tid < n_terms) {
    const PanelTerm tm = terms[pt.term0 + tid];
    const double2 v = ld_elem<E, CPLX>(B + tm.b * P);
    s_br[tid] = v.x;
    s_bi[tid] = v.y;
  } else if (tid >= 128 && tid < 128 + n_outs) {
    const int o = tid - 128;
    const PanelOut po = outs[pt.out0 + o];
    const Seg &sg = segs[po.seg];
    s_ocoff[o] = sg.c_off + po.j;
    s_on[o] = sg.n;
    s_ot0[o] = po.term0;
    s_omask[o] = po.mask;
  }
  __syncthreads();
  // the paired columns of this thread's rows
#pragma unroll
  for (int c = 0; c < kPanelCols; ++c)
    if (pc >= 0 && (c == pc || c == pc + 1)) {
      const int cc = c - pc;
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        av[c][q] = s_pa[cc][tid + 256 * q];
        av_i[c][q] = CPLX ? s_pai[CPLX ? cc : 0][tid + 256 * q] : 0.0;
      }
    }

  // The output loop exists twice, for beta == 0 and beta != 0: with the
  // loads of the old values inside a shared loop, every output column waited
  // for the previous column's stores (stores count in the same counter).
  auto out_loop = [&](auto with_beta) {
    constexpr bool WB = decltype(with_beta)::value;
    for (int o = 0; o < n_outs; ++o) {
      const int64_t coff = s_ocoff[o];
      const int32_t n = __builtin_amdgcn_readfirstlane(s_on[o]);
      const int32_t mask = __builtin_amdgcn_readfirstlane(s_omask[o]);
      int32_t t = __builtin_amdgcn_readfirstlane(s_ot0[o]);
      double y[RPT], y_i[RPT];
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        y[q] = 0.0;
        y_i[q] = 0.0;
      }
      // the output's terms in ascending column order, which is their (task, k)
      // order: the column loop is static, so no register array is indexed
#pragma unroll
      for (int c = 0; c < kPanelCols; ++c) {
        if (!((mask >> c) & 1)) continue;
        const double b = s_br[t], b_im = s_bi[t];
        ++t;
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
          if (CPLX) {
            y[q] = fma(av[c][q], b, y[q]);
            y[q] = fma(-av_i[c][q], b_im, y[q]);
            y_i[q] = fma(av[c][q], b_im, y_i[q]);
            y_i[q] = fma(av_i[c][q], b, y_i[q]);
          } else {
            y[q] = fma(av[c][q], b, y[q]);
          }
        }
      }
      raw_t<E, CPLX> old[RPT] = {};
      if constexpr (WB) {
#pragma unroll
        for (int q = 0; q < RPT; ++q)
          old[q] = ld_raw<E, CPLX>(C + P * (coff + (valid[q] ? static_cast<int64_t>(pt.r0 + tid + 256 * q) * n : 0)));
      }
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        if (!valid[q]) continue;
        const int64_t e = coff + static_cast<int64_t>(pt.r0 + tid + 256 * q) * n;
        st_scaled<E, CPLX>(C + P * e, y[q], CPLX ? y_i[q] : 0.0, old[q], WB, alpha_r, alpha_i, beta_r, beta_i);
      }
    }
  };
  if (beta_r != 0.0 || beta_i != 0.0) out_loop(std::true_type{});
  else out_loop(std::false_type{});
}

// ---- kernels: one tile class, or all classes of a contraction ----

// What every kernel of a contraction reads; tiles and reduction items are
// stored class-major, and each class has its own region of `part`.
template <typename E>
struct ExecArgs {
  const Tile *tiles;
  const ReduceItem *red;
  const Seg *segs;
  const ExecTask *exec;
  const BlkGather *ga, *gb;
  const PanelTile *ptiles;
  const PanelOut *pouts;
  const PanelTerm *pterms;
  const E *A, *B;
  E *C;
  double *part;
  double ar, ai, br, bi;
  GatherLayout L;
  int64_t part_off[kNumTileClasses];
  int32_t tile0[kNumTileClasses];     // first tile of the class
  int32_t count[kNumTileClasses];     // its tiles
  int32_t block0[kNumTileClasses + 1];  // k_all_classes: first workgroup of the class, and of the panels
};

// Order of the classes in k_all_classes: the few narrow-output tiles, whose
// chains of contracted indices are the longest, start first.
constexpr int32_t kLaunchOrder[] = {kTileNarrow, kTileRows4, 1, 3, kNumTileClasses};

// Workgroup `b` of `n` of class CLS.
template <bool CPLX, int CLS, typename E>
__device__ __forceinline__ void class_block(char *smem, const ExecArgs<E> &x, int b, int n,
                                            const Tile *__restrict__ tiles, const Seg *__restrict__ segs,
                                            const ExecTask *__restrict__ exec, const BlkGather *__restrict__ ga,
                                            const BlkGather *__restrict__ gb, const E *__restrict__ A,
                                            const E *__restrict__ B, E *__restrict__ C, double *__restrict__ part) {
  const Tile tile = tiles[x.tile0[CLS] + xcd_tile(b, n)];
  double *const cp = part + x.part_off[CLS];
  if constexpr (CLS == kTileRows4)
    rows_tile<CPLX, 4, 4, E>(smem, tile, segs, exec, ga, gb, x.L, A, B, C, cp, x.ar, x.ai, x.br, x.bi);
  else if constexpr (CLS == kTileNarrowRows)
    narrow_tile<CPLX, 1, E>(smem, tile, segs, exec, ga, gb, x.L, A, B, C, cp, x.ar, x.ai, x.br, x.bi);
  else if constexpr (CLS == kTileNarrow)
    narrow_tile<CPLX, kNarrowWaves, E>(smem, tile, segs, exec, ga, gb, x.L, A, B, C, cp, x.ar, x.ai, x.br, x.bi);
  else
    grouped_tile<CPLX, mfma_tile_m(CLS), mfma_tile_n(CLS), E>(smem, tile, segs, exec, ga, gb, x.L, A, B, C, cp, x.ar,
                                                              x.ai, x.br, x.bi);
}
template <bool CPLX, int CLS>
constexpr size_t class_shared() {
  if constexpr (CLS == kTileRows4) return sizeof(RowsShared<CPLX, 4>);
  else if constexpr (CLS == kTileNarrow) return sizeof(NarrowShared<CPLX>);
  else if constexpr (CLS == kTileNarrowRows) return 16;
  else return sizeof(GroupedShared<CPLX, mfma_tile_m(CLS), mfma_tile_n(CLS)>);
}

template <bool CPLX, int CLS, typename E>
__global__ __launch_bounds__(256) void k_class(const ExecArgs<E> x) {
  __shared__ __align__(16) char smem[class_shared<CPLX, CLS>()];
  class_block<CPLX, CLS, E>(smem, x, static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x), x.tiles, x.segs, x.exec,
                            x.ga, x.gb, x.A, x.B, x.C, x.part);
}
// The row classes, whose pointers are restrict-qualified arguments of their
// own: read from a struct they may alias the output as far as the compiler
// knows, and the per-task descriptors came by vector loads, each waited for,
// instead of scalar ones (n = 4, k = 5, m = 1000 in FP64: 7.0 -> 5.3 us).
template <bool CPLX, int CLS, typename E>
__global__ __launch_bounds__(256) void k_row_class(const ExecArgs<E> x, const Tile *__restrict__ tiles,
                                                   const Seg *__restrict__ segs, const ExecTask *__restrict__ exec,
                                                   const BlkGather *__restrict__ ga, const BlkGather *__restrict__ gb,
                                                   const E *__restrict__ A, const E *__restrict__ B,
                                                   E *__restrict__ C, double *__restrict__ part) {
  __shared__ __align__(16) char smem[class_shared<CPLX, CLS>()];
  class_block<CPLX, CLS, E>(smem, x, static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x), tiles, segs, exec, ga,
                            gb, A, B, C, part);
}
template <bool CPLX, bool STREAM, typename E>
__global__ __launch_bounds__(256) void k_panel_rows(const ExecArgs<E> x) {
  __shared__ __align__(16) char smem[sizeof(PanelShared<CPLX>)];
  panel_tile<CPLX, STREAM, E>(smem, x.ptiles[blockIdx.x], x.pouts, x.pterms, x.segs, x.A, x.B, x.C, x.ar, x.ai, x.br,
                              x.bi);
}
// Every class of a contraction in one launch (the 64-row MFMA classes, which
// only a tuning table selects, excepted).  With a launch per class on streams
// forked from the caller's and joined back, the forks and the gaps between
// dependent launches were most of a small contraction and a tenth of a large
// one: U(1) FP64 matvec at D = 96 103 -> 32 us, D = 700 164 -> 43 us, lognormal
// 184 -> 117 us, U(1)xU(1) complex128 D = 1500 252 -> 156 us, D = 4096 1.22 ->
// 1.18 ms.  The register bound keeps the occupancy of the widest class alone
// (complex: three workgroups per CU; unbounded, two, and D = 4096 took 1.35 ms;
// real: five, with D = 2048 FP64 285 -> 272 us from four; six spill).  The
// row and grouped classes read through the restrict-qualified arguments, as in
// k_row_class (D = 2048 FP64 matvec 273.9 -> 273.3 us, D = 4096 complex128
// 1.116 -> 1.101 ms); the n <= 16 tiles, a chain of few loads, through the struct
// (complex64 accumulate 49.7 us, 51.3 with scalar loads on the chain).
template <bool CPLX, bool STREAM, typename E>
__global__ __launch_bounds__(256, CPLX ? 3 : 5) void k_all_classes(
    const ExecArgs<E> x, const Tile *__restrict__ tiles, const Seg *__restrict__ segs,
    const ExecTask *__restrict__ exec, const BlkGather *__restrict__ ga, const BlkGather *__restrict__ gb,
    const E *__restrict__ A, const E *__restrict__ B, E *__restrict__ C, double *__restrict__ part) {
  constexpr size_t kBytes = std::max({class_shared<CPLX, 1>(), class_shared<CPLX, 3>(), class_shared<CPLX, 4>(),
                                      class_shared<CPLX, 6>(), sizeof(PanelShared<CPLX>)});
  __shared__ __align__(16) char smem[kBytes];
  const int b = static_cast<int>(blockIdx.x);
  if (b < x.block0[4])
    class_block<CPLX, 6, E>(smem, x, b - x.block0[6], x.count[6], x.tiles, x.segs, x.exec, x.ga, x.gb, x.A, x.B, x.C,
                            x.part);
  else if (b < x.block0[1])
    class_block<CPLX, 4, E>(smem, x, b - x.block0[4], x.count[4], tiles, segs, exec, ga, gb, A, B, C, part);
  else if (b < x.block0[3])
    class_block<CPLX, 1, E>(smem, x, b - x.block0[1], x.count[1], tiles, segs, exec, ga, gb, A, B, C, part);
  else if (b < x.block0[7])
    class_block<CPLX, 3, E>(smem, x, b - x.block0[3], x.count[3], tiles, segs, exec, ga, gb, A, B, C, part);
  else
    panel_tile<CPLX, STREAM, E>(smem, x.ptiles[b - x.block0[7]], x.pouts, x.pterms, segs, A, B, C, x.ar, x.ai, x.br,
                                x.bi);
}
// The k-slice sums of reduction items first, first + 1, ...
template <bool CPLX, typename E>
__global__ __launch_bounds__(256) void k_reduce(const ExecArgs<E> x, int first) {
  const ReduceItem it = x.red[first + static_cast<int>(blockIdx.x)];
  const Seg seg = x.segs[it.seg];
  const double *part = x.part + x.part_off[it.cls];
  switch (it.cls) {
    case 0: reduce_slices<CPLX, 64, 64, E>(it, seg, part, x.C, x.ar, x.ai, x.br, x.bi); break;
    case 1: reduce_slices<CPLX, 32, 64, E>(it, seg, part, x.C, x.ar, x.ai, x.br, x.bi); break;
    case 2: reduce_slices<CPLX, 64, 32, E>(it, seg, part, x.C, x.ar, x.ai, x.br, x.bi); break;
    case 3: reduce_slices<CPLX, 32, 32, E>(it, seg, part, x.C, x.ar, x.ai, x.br, x.bi); break;
    case kTileRows4: reduce_rows<CPLX, 4, 4, E>(it, seg, part, x.C, x.ar, x.ai, x.br, x.bi); break;
    case kTileNarrowRows: reduce_slices<CPLX, kNarrowM * kNarrowWaves, kNarrowN, E>(it, seg, part, x.C, x.ar, x.ai, x.br, x.bi); break;
    default: reduce_slices<CPLX, kNarrowM, kNarrowN, E>(it, seg, part, x.C, x.ar, x.ai, x.br, x.bi); break;
  }
}

}  // namespace

namespace qlt {

// Native grouped execution of a plan.  `mfma_class` = false leaves out the
// MFMA classes with n > 16 (the split path runs them on its own kernel).
qlt_status launch_native_classes(const qlt_plan *plan, int32_t dtype, const void *a, const void *b, void *c,
                                 const double *alpha, const double *beta, hipStream_t st, bool mfma_class,
                                 bool probe, ClassStreams *shared) {
  const bool cplx = dtype_is_complex(dtype);
  constexpr int32_t kPanelId = kNumTileClasses;
  // the classes this call runs, the panels last
  auto runs = [&](int32_t cls) {
    if (cls == kPanelId) return plan->n_ptiles > 0;
    return plan->cls_tiles[cls] > 0 && (mfma_class || !is_mfma_class(cls));
  };
  int n_cls = 0;
  for (int32_t cls = 0; cls <= kPanelId; ++cls) n_cls += runs(cls);
  if (n_cls == 0) return QLT_OK;
  // the class with the most algorithmic work is the one a kernel probe times,
  // in a launch of its own
  int32_t dom = -1;
  if (probe && probe_armed(st)) {
    double best = 0.0;
    for (int32_t cls = 0; cls < kNumTileClasses; ++cls)
      if (runs(cls) && plan->cls_mkn[cls] > best) {
        best = plan->cls_mkn[cls];
        dom = cls;
      }
    if (runs(kPanelId) && plan->panel_mkn > best) dom = kPanelId;
  }
  // One stream, and one launch for the classes that k_all_classes holds; a
  // probed class, and the 64-row classes, take a launch per class on the class
  // streams.  The kTileNarrowRows class fills the chip by itself and has a launch of
  // its own before the others'.  A launch holds less than 2^32 threads.
  const bool one_stream = dom < 0 && !runs(0) && !runs(2);
  const bool fused = one_stream && n_cls - (runs(kTileNarrowRows) ? 1 : 0) >= 2 &&
                     plan->n_tiles + plan->n_ptiles < (int64_t(1) << 24);
  std::unique_ptr<ClassStreams> own;
  ClassStreams *cs = shared;
  if (cs == nullptr && n_cls >= 2 && !one_stream) {
    own = std::make_unique<ClassStreams>(st);
    cs = own.get();
  }
  auto stream_of = [&](int32_t cls) {
    if (cls == kPanelId || one_stream) cls = kTileRows4;
    return cs != nullptr ? cs->get(cls) : st;
  };
  auto probe_in = [&](int32_t cls) {
    if (cls == dom) probe_begin(stream_of(cls));
  };
  auto probe_out = [&](int32_t cls) {
    if (cls != dom) return;
    const hipStream_t ps = stream_of(cls);
    // the n <= 16 class keeps the name of the row class it is
    static const char *const kNames[kNumTileClasses + 1] = {
        "k_grouped_gemm_f64<64x64>", "k_grouped_gemm_f64<32x64>", "k_grouped_gemm_f64<64x32>",
        "k_grouped_gemm_f64<32x32>", "k_rows_f64<n<=4>",          "k_rows_f64<n<=16>",
        "k_rows_f64<n<=16>",          "k_panel_rows"};
    char name[64];
    static const char *const kTypes[4] = {"f64", "c128", "f32", "c64"};
    std::snprintf(name, sizeof(name), "%s %s", kNames[cls], kTypes[dtype & 3]);
    const double mkn = cls == kPanelId ? plan->panel_mkn : plan->cls_mkn[cls];
    const double elems = cls == kPanelId ? plan->panel_elems : plan->cls_elems[cls];
    probe_end(ps, name, (cplx ? 8.0 : 2.0) * mkn, static_cast<double>(dtype_bytes(dtype)) * elems);
  };
  const dim3 block(256);
  auto grid_of = [](int64_t n) { return dim3(static_cast<unsigned>(n)); };
  // every kernel instance of one element storage type E (double, or float
  // for the single-precision element types) and complexity
  auto run = [&](auto e_tag, auto cplx_tag) {
    using E = decltype(e_tag);
    constexpr bool CX = decltype(cplx_tag)::value;
    ExecArgs<E> x{};
    x.tiles = plan->d_tiles;
    x.red = plan->d_red;
    x.segs = plan->d_segs;
    x.exec = plan->d_exec;
    x.ga = plan->d_ga;
    x.gb = plan->d_gb;
    x.ptiles = plan->d_ptiles;
    x.pouts = plan->d_pouts;
    x.pterms = plan->d_pterms;
    x.A = static_cast<const E *>(a);
    x.B = static_cast<const E *>(b);
    x.C = static_cast<E *>(c);
    x.part = plan->d_part;
    x.ar = alpha[0];
    x.ai = CX ? alpha[1] : 0.0;
    x.br = beta[0];
    x.bi = CX ? beta[1] : 0.0;
    x.L = plan->layout;
    int64_t base = 0, red_base = 0;
    int32_t red0[kNumTileClasses];
    int64_t first_red = -1, n_red = 0;
    for (int32_t cls = 0; cls < kNumTileClasses; ++cls) {
      x.part_off[cls] = plan->cls_part_off[cls];
      x.tile0[cls] = static_cast<int32_t>(base);
      x.count[cls] = static_cast<int32_t>(plan->cls_tiles[cls]);
      red0[cls] = static_cast<int32_t>(red_base);
      if (runs(cls) && plan->cls_red[cls] > 0) {
        if (first_red < 0) first_red = red_base;
        n_red = red_base + plan->cls_red[cls] - first_red;   // the classes that run are the last ones: contiguous
      }
      base += plan->cls_tiles[cls];
      red_base += plan->cls_red[cls];
    }
    int64_t blocks = 0;
    for (const int32_t cls : kLaunchOrder) {
      x.block0[cls] = static_cast<int32_t>(blocks);
      if (cls == kPanelId) blocks += plan->n_ptiles;
      else if (runs(cls)) blocks += plan->cls_tiles[cls];
    }
    // non-temporal A' loads only when the panels' A' and C exceed the
    // last-level cache: smaller ones are served from it (measured: a
    // 0.83 GB W contraction 0.169 -> 0.148 ms with the hint, a small one
    // 0.028 -> 0.032 ms)
    const bool stream_a = plan->panel_elems * static_cast<double>(sizeof(E) * (CX ? 2 : 1)) > kPanelStreamBytes;
    auto one = [&](auto cls_tag) {
      constexpr int CLS = decltype(cls_tag)::value;
      if (!runs(CLS)) return;
      const hipStream_t ls = stream_of(CLS);
      probe_in(CLS);
      if constexpr (CLS == kTileRows4)
        hipLaunchKernelGGL((k_row_class<CX, CLS, E>), grid_of(plan->cls_tiles[CLS]), block, 0, ls, x, x.tiles, x.segs,
                           x.exec, x.ga, x.gb, x.A, x.B, x.C, x.part);
      else hipLaunchKernelGGL((k_class<CX, CLS, E>), grid_of(plan->cls_tiles[CLS]), block, 0, ls, x);
      probe_out(CLS);
      // k-sliced tiles: the slices wrote partial sums; one workgroup per sliced
      // tile adds them and applies alpha / beta
      if (!fused && plan->cls_red[CLS] > 0)
        hipLaunchKernelGGL((k_reduce<CX, E>), grid_of(plan->cls_red[CLS]), block, 0, ls, x, red0[CLS]);
    };
    one(std::integral_constant<int, kTileNarrowRows>{});
    if (fused) {
      const hipStream_t ls = stream_of(kTileRows4);
      const auto kernel = stream_a ? k_all_classes<CX, true, E> : k_all_classes<CX, false, E>;
      hipLaunchKernelGGL(kernel, grid_of(blocks), block, 0, ls, x, x.tiles, x.segs, x.exec, x.ga, x.gb, x.A, x.B, x.C,
                         x.part);
      if (n_red > 0) hipLaunchKernelGGL((k_reduce<CX, E>), grid_of(n_red), block, 0, ls, x, static_cast<int>(first_red));
      return;
    }
    one(std::integral_constant<int, 0>{});
    one(std::integral_constant<int, 1>{});
    one(std::integral_constant<int, 2>{});
    one(std::integral_constant<int, 3>{});
    one(std::integral_constant<int, kTileRows4>{});
    one(std::integral_constant<int, kTileNarrow>{});
    // row panels, after the n <= 4 row class on its stream
    if (runs(kPanelId)) {
      const hipStream_t ls = stream_of(kPanelId);
      probe_in(kPanelId);
      if (stream_a) hipLaunchKernelGGL((k_panel_rows<CX, true, E>), grid_of(plan->n_ptiles), block, 0, ls, x);
      else hipLaunchKernelGGL((k_panel_rows<CX, false, E>), grid_of(plan->n_ptiles), block, 0, ls, x);
      probe_out(kPanelId);
    }
  };
  switch (dtype) {
    case QLT_F64: run(double{}, std::false_type{}); break;
    case QLT_C128: run(double{}, std::true_type{}); break;
    case QLT_F32: run(float{}, std::false_type{}); break;
    default: run(float{}, std::true_type{}); break;
  }
  QLT_HIP(hipGetLastError());
  return QLT_OK;
}

qlt_status launch_native(const qlt_plan *plan, int32_t dtype, const void *a, const void *b, void *c,
                         const double *alpha, const double *beta, hipStream_t st) {
  return launch_native_classes(plan, dtype, a, b, c, alpha, beta, st, true, true, nullptr);
}

}  // namespace qlt
