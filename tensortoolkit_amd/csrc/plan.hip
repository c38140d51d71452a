// Contraction plan building.
//
// Reproduces BlockSparseDataTensor::DataBlkGenForTenCtrct
// (include/qlten/qltensor/blk_spar_data_ten/data_blk_operations.h:411-578)
// bit for bit, by integer arithmetic:
//   1. part hash of each block's contracted coordinates, taken in the given
//      axis order (VecPartHasher, include/qlten/framework/vec_hash.h:39-47,
//      via GenBlkIdxQNBlkCoorPartHashMap, blk_spar_data_ten.h:959-973);
//   2. A-major / B-minor matching on equal hashes, both in ascending block
//      index (data_blk_operations.h:494-567); for a scalar output the B loop
//      stops at the first match (data_blk_operations.h:451-491);
//   3. output block creation on first touch -> beta 0, later touches beta 1;
//   4. output offsets = exclusive prefix sum of block sizes in ascending
//      output block index (DataBlksOffsetRefresh, data_blk_operations.h:137-145,568);
//   5. c_data_offset fill (data_blk_operations.h:571-574).
// The device finds the tasks (1, 2) and sorts them by output block (an order
// SortTasksByCBlkIdx, raw_data_operation_tasks.h:250-269, can produce, with
// generation order kept inside a block); the host reads back 20 bytes per task
// and fills the records that are linear in the tasks: task fields, output
// blocks and offsets (3 - 5), and the grouped-GEMM work list -- one segment per
// output block, its tiles longest first, k-slices and row panels -- which goes
// to the device in one copy.
//   What bounds it is latency: launches and copies of a few microseconds each
// around little work.  Every array on the device came back in a copy of its
// own, the gather descriptors twice, and each tile list was built, sorted, read
// back, re-cut and uploaded again.  Per plan: U(1) FP64, 139 tasks, 480 -> 105 us;
// U(1)xU(1) D = 512, 4860 tasks, 1180 -> 430 us.

#include <algorithm>
#include <atomic>
#include <memory>
#include <cstring>
#include <numeric>
#include <string>

#include "qlt_internal.h"

using namespace qlt;

namespace {

constexpr uint64_t kP1 = 11400714785074694791ull;
constexpr uint64_t kP2 = 14029467366897019727ull;
constexpr uint64_t kP5 = 2870177450012600261ull;

struct PlanArgs {
  int32_t a_rank, b_rank, n_ctrct, n_a_saved, n_b_saved, c_rank;
  int32_t a_ctrct[QLT_MAX_RANK], b_ctrct[QLT_MAX_RANK];
  int32_t a_saved[QLT_MAX_RANK], b_saved[QLT_MAX_RANK];
  int64_t c_stride[QLT_MAX_RANK];
  int32_t c_is_scalar;
  int8_t cls_table[QLT_TUNE_BUCKETS][QLT_TUNE_BUCKETS];   // tile class per size bucket (qlt_tuning)
};

struct DevTask {
  int32_t a_pos;
  int32_t b_pos;
};

__device__ __forceinline__ uint64_t rotl31(uint64_t x) { return (x << 31) | (x >> 33); }

// Hashes of both operands' blocks: A's in h[0 .. na), B's in h[na .. na + nb).
__global__ void k_part_hash(const int32_t *a_coords, int64_t na, const int32_t *b_coords, int64_t nb,
                            const PlanArgs args, uint64_t *h) {
  const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i >= na + nb) return;
  const bool is_a = i < na;
  const int32_t *c = is_a ? a_coords + i * args.a_rank : b_coords + (i - na) * args.b_rank;
  const int32_t *axes = is_a ? args.a_ctrct : args.b_ctrct;
  uint64_t hv = kP5;
  for (int j = 0; j < args.n_ctrct; ++j) {
    hv += static_cast<uint64_t>(c[axes[j]]) * kP2;
    hv = rotl31(hv);
    hv *= kP1;
  }
  hv += static_cast<uint64_t>(args.n_ctrct) ^ kP5;
  h[i] = hv;
}

// counts[i] = number of B blocks whose hash equals A block i's (at most 1 for
// a scalar output).  B hashes are staged through LDS.
__global__ __launch_bounds__(256) void k_count(const uint64_t *ha, int64_t na, const uint64_t *hb,
                                               int64_t nb, int32_t scalar, int64_t *counts) {
  __shared__ uint64_t sh[1024];
  const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  const uint64_t mine = (i < na) ? ha[i] : 0;
  int64_t cnt = 0;
  for (int64_t base = 0; base < nb; base += 1024) {
    const int64_t len = (nb - base < 1024) ? (nb - base) : 1024;
    __syncthreads();
    for (int64_t j = threadIdx.x; j < len; j += blockDim.x) sh[j] = hb[base + j];
    __syncthreads();
    if (i < na)
      for (int64_t j = 0; j < len; ++j) cnt += (sh[j] == mine) ? 1 : 0;
  }
  if (i < na) counts[i] = (scalar && cnt > 1) ? 1 : cnt;
}

// Single-workgroup exclusive scan of n int64 values; total written to *total.
__global__ __launch_bounds__(1024) void k_scan_excl(const int64_t *in, int64_t *out, int64_t n,
                                                    int64_t *total) {
  __shared__ int64_t wsum[16];
  __shared__ int64_t carry;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  if (tid == 0) carry = 0;
  __syncthreads();
  for (int64_t base = 0; base < n; base += 1024) {
    const int64_t i = base + tid;
    const int64_t v = (i < n) ? in[i] : 0;
    int64_t x = v;
    for (int off = 1; off < 64; off <<= 1) {
      const int64_t y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int64_t wprefix = 0;
    for (int j = 0; j < w; ++j) wprefix += wsum[j];
    const int64_t c = carry;
    if (i < n) out[i] = c + wprefix + x - v;
    __syncthreads();
    if (tid == 1023) carry = c + wprefix + x;
    __syncthreads();
  }
  if (tid == 0) *total = carry;
}

// One wavefront per A block: walk B in ascending order, ballot the matches
// and write them at consecutive task slots, so the task list comes out in
// the reference's A-major / B-minor order; with each task its output block
// index (the sort key), its position (the payload of the radix sort) and a
// cleared rank.
__global__ __launch_bounds__(256) void k_emit(const uint64_t *ha, int64_t na, const uint64_t *hb, int64_t nb,
                                              const int64_t *starts, const int32_t *a_coords, const int32_t *b_coords,
                                              const PlanArgs args, DevTask *tasks, uint64_t *key, int32_t *val,
                                              int32_t *rank) {
  const int lane = threadIdx.x & 63;
  const int64_t i = (blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x) >> 6;
  if (i >= na) return;
  const uint64_t mine = ha[i];
  const int32_t *ac = a_coords + i * args.a_rank;
  uint64_t ka = 0;
  if (!args.c_is_scalar)
    for (int j = 0; j < args.n_a_saved; ++j)
      ka += static_cast<uint64_t>(ac[args.a_saved[j]]) * static_cast<uint64_t>(args.c_stride[j]);
  auto put = [&](int64_t t, int64_t j) {
    uint64_t k = ka;
    if (!args.c_is_scalar) {
      const int32_t *bc = b_coords + j * args.b_rank;
      for (int q = 0; q < args.n_b_saved; ++q)
        k += static_cast<uint64_t>(bc[args.b_saved[q]]) * static_cast<uint64_t>(args.c_stride[args.n_a_saved + q]);
    }
    tasks[t] = DevTask{static_cast<int32_t>(i), static_cast<int32_t>(j)};
    key[t] = k;
    val[t] = static_cast<int32_t>(t);
    rank[t] = 0;
  };
  int64_t pos = starts[i];
  for (int64_t base = 0; base < nb; base += 64) {
    const int64_t j = base + lane;
    const bool match = (j < nb) && (hb[j] == mine);
    const uint64_t bal = __ballot(match);
    if (bal == 0) continue;
    if (args.c_is_scalar) {
      const int first = __ffsll(static_cast<unsigned long long>(bal)) - 1;
      if (lane == first) put(pos, j);
      return;
    }
    const int before = __popcll(bal & ((1ull << lane) - 1ull));
    if (match) put(pos + before, j);
    pos += __popcll(bal);
  }
}

// Sorted position of every task by counting: rank[t] = tasks of smaller key,
// plus tasks of equal key before t.  Grid (256 tasks, chunk of kRankChunk keys
// to compare them with).  Quadratic, but spread over the chip: up to
// kRankMaxTasks it is faster than the single-workgroup radix sort (43 us at
// 4860 tasks, 170 us at 45 000).  What bounds it is the LDS latency of the keys
// (one address for the whole wave), so the comparisons run in groups whose
// keys are read together, with no test of the position but in the chunk on the
// diagonal: 52 -> 7.6 us at 4600 tasks, 54 -> 11.9 at 11 500 (chunks of 1024
// and a loop over each side of the position before).
constexpr int kRankChunk = 256;
constexpr int64_t kRankMaxTasks = 32768;
__global__ __launch_bounds__(256) void k_rank(const uint64_t *key, int64_t n, int32_t *rank) {
  __shared__ __align__(16) uint64_t sk[kRankChunk];
  static_assert(kRankChunk == 256, "a chunk per workgroup of tasks: one key per thread");
  const int tid = threadIdx.x;
  const int64_t base = int64_t(blockIdx.y) * kRankChunk, t = int64_t(blockIdx.x) * 256 + tid;
  sk[tid] = base + tid < n ? key[base + tid] : ~uint64_t(0);   // past the end: never smaller
  const uint64_t mine = t < n ? key[t] : 0;
  __syncthreads();
  int32_t r = 0;
  if (blockIdx.y < blockIdx.x) {   // keys before position t count when equal, too
#pragma unroll 16
    for (int j = 0; j < kRankChunk; ++j) r += sk[j] <= mine ? 1 : 0;
  } else if (blockIdx.y > blockIdx.x) {
#pragma unroll 16
    for (int j = 0; j < kRankChunk; ++j) r += sk[j] < mine ? 1 : 0;
  } else {
#pragma unroll 16
    for (int j = 0; j < kRankChunk; ++j) r += sk[j] < mine + (j < tid ? 1 : 0) ? 1 : 0;
  }
  if (t < n && r != 0) atomicAdd(&rank[t], r);
}
__global__ void k_place(const uint64_t *key, const int32_t *rank, int64_t n, uint64_t *sk, int32_t *sv) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (t >= n) return;
  sk[rank[t]] = key[t];
  sv[rank[t]] = static_cast<int32_t>(t);
}

// Single-workgroup stable LSD radix sort (8-bit digits) of (key, val) pairs.
// Each 1024-element chunk is ranked with a wavefront multisplit (eight
// ballots per element) and chunks are placed in input order, so equal keys
// keep their input order.  The result is in (k0, v0) after an even number of
// passes and in (k1, v1) after an odd one.
__global__ __launch_bounds__(1024) void k_radix_sort(uint64_t *k0, int32_t *v0, uint64_t *k1,
                                                     int32_t *v1, int64_t n, int32_t passes) {
  __shared__ int64_t digit_base[256];
  __shared__ int32_t chunk_cnt[256];
  __shared__ int32_t wave_cnt[16][256];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int pass = 0; pass < passes; ++pass) {
    const uint64_t *sk = (pass & 1) ? k1 : k0;
    const int32_t *sv = (pass & 1) ? v1 : v0;
    uint64_t *dk = (pass & 1) ? k0 : k1;
    int32_t *dv = (pass & 1) ? v0 : v1;
    const int shift = 8 * pass;
    if (tid < 256) chunk_cnt[tid] = 0;
    __syncthreads();
    for (int64_t i = tid; i < n; i += 1024) atomicAdd(&chunk_cnt[(sk[i] >> shift) & 255u], 1);
    __syncthreads();
    if (tid == 0) {
      int64_t run = 0;
      for (int d = 0; d < 256; ++d) {
        digit_base[d] = run;
        run += chunk_cnt[d];
      }
    }
    __syncthreads();
    for (int64_t chunk = 0; chunk < n; chunk += 1024) {
      const int64_t i = chunk + tid;
      const bool valid = i < n;
      const uint64_t key = valid ? sk[i] : 0;
      const int32_t val = valid ? sv[i] : 0;
      const int d = static_cast<int>((key >> shift) & 255u);
      for (int j = tid; j < 16 * 256; j += 1024) wave_cnt[j >> 8][j & 255] = 0;
      __syncthreads();
      uint64_t mask = __ballot(valid);
      for (int b = 0; b < 8; ++b) {
        const bool bit = (d >> b) & 1;
        const uint64_t bal = __ballot(bit);
        mask &= bit ? bal : ~bal;
      }
      const int rank = __popcll(mask & ((1ull << lane) - 1ull));
      if (valid && rank == 0) wave_cnt[w][d] = __popcll(mask);
      __syncthreads();
      if (tid < 256) {
        int32_t run = 0;
        for (int ww = 0; ww < 16; ++ww) {
          const int32_t c = wave_cnt[ww][tid];
          wave_cnt[ww][tid] = run;
          run += c;
        }
        chunk_cnt[tid] = run;
      }
      __syncthreads();
      if (valid) {
        const int64_t pos = digit_base[d] + wave_cnt[w][d] + rank;
        dk[pos] = key;
        dv[pos] = val;
      }
      __syncthreads();
      if (tid < 256) digit_base[tid] += chunk_cnt[tid];
      __syncthreads();
    }
  }
}

// The permuted view of one input block: A blocks are read as (saved ++
// contracted), B blocks as (contracted ++ saved).  Row (col) axis j has extent
// rdim[j] and memory stride rstr[j] (cdim, cstr).
struct BlkShape {
  int32_t rdim[QLT_MAX_RANK], rstr[QLT_MAX_RANK], cdim[QLT_MAX_RANK], cstr[QLT_MAX_RANK];
  int32_t nrows, ncols;
  int32_t plain;         // the view is the block itself in memory order
  int32_t fastcol;       // the block's innermost axis of extent > 1 (stride 1) is a col axis
  int32_t caff, cstep;   // the col (row) axes of extent > 1 merge into one
  int32_t raff, rstep;
};
__host__ __device__ inline void blk_shape(const int32_t *d, int32_t rank, const int32_t *raxes, int32_t nr,
                                          const int32_t *caxes, int32_t nc, BlkShape &g) {
  int32_t stride[QLT_MAX_RANK];
  int32_t s = 1, inner = -1;
  for (int j = rank - 1; j >= 0; --j) {
    stride[j] = s;
    s *= d[j];
    if (inner < 0 && d[j] > 1) inner = j;
  }
  int32_t last_axis = -1;
  g.plain = 1;
  g.fastcol = 0;
  // one part's axes; affine when every adjacent pair of axes of extent > 1
  // satisfies stride[j] == stride[j + 1] * dim[j + 1]
  auto part = [&](const int32_t *axes, int n, int32_t *dim, int32_t *str, int32_t &total, int32_t &aff, int32_t &step) {
    int32_t last = -1;
    total = 1;
    aff = 1;
    step = 1;
    for (int j = 0; j < n; ++j) {
      const int32_t ax = axes[j];
      dim[j] = d[ax];
      str[j] = stride[ax];
      total *= d[ax];
      if (d[ax] <= 1) continue;
      if (ax < last_axis) g.plain = 0;
      last_axis = ax;
      if (last >= 0 && str[last] != str[j] * dim[j]) aff = 0;
      last = j;
    }
    if (last >= 0) step = str[last];
  };
  part(raxes, nr, g.rdim, g.rstr, g.nrows, g.raff, g.rstep);
  part(caxes, nc, g.cdim, g.cstr, g.ncols, g.caff, g.cstep);
  for (int j = 0; j < nc; ++j)
    if (caxes[j] == inner) g.fastcol = 1;
}

// Gather descriptors of A's blocks (out_a) and B's (out_b), 2 QLT_MAX_RANK
// threads per block: one axis of one part each, whose reciprocal is the
// kernel's chain (one thread per block took 14 us).
__global__ void k_gather_desc(const int32_t *a_dims, int64_t na, const int32_t *b_dims, int64_t nb,
                              const PlanArgs args, BlkGather *out_a, BlkGather *out_b) {
  const int64_t gid = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  const int64_t i = gid / (2 * QLT_MAX_RANK);
  const int part = static_cast<int>(gid % (2 * QLT_MAX_RANK)), j = part % QLT_MAX_RANK;
  if (i >= na + nb) return;
  const bool is_a = i < na;
  const int32_t nr = is_a ? args.n_a_saved : args.n_ctrct, nc = is_a ? args.n_ctrct : args.n_b_saved;
  BlkShape v;
  if (is_a) blk_shape(a_dims + i * args.a_rank, args.a_rank, args.a_saved, nr, args.a_ctrct, nc, v);
  else blk_shape(b_dims + (i - na) * args.b_rank, args.b_rank, args.b_ctrct, nr, args.b_saved, nc, v);
  BlkGather &g = is_a ? out_a[i] : out_b[i - na];
  int32_t dim = 1, str = 0;
#pragma unroll
  for (int q = 0; q < QLT_MAX_RANK; ++q) {   // constant indexes keep v in registers
    if (part < QLT_MAX_RANK && q == j && j < nr) {
      dim = v.rdim[q];
      str = v.rstr[q];
    }
    if (part >= QLT_MAX_RANK && q == j && j < nc) {
      dim = v.cdim[q];
      str = v.cstr[q];
    }
  }
  uint64_t mag;
  int32_t sh;
  magic_of(static_cast<uint32_t>(dim), mag, sh);
  if (part < QLT_MAX_RANK) {
    g.rdim[j] = dim;
    g.rstr[j] = str;
    g.rmag[j] = mag;
    g.rsh[j] = sh;
  } else {
    g.cdim[j] = dim;
    g.cstr[j] = str;
    g.cmag[j] = mag;
    g.csh[j] = sh;
  }
  if (part == 0) {
    g.plain = v.plain;
    g.ncols = v.ncols;
    g.nrows = v.nrows;
    g.fastcol = v.fastcol;
    g.caff = v.caff;
    g.cstep = v.cstep;
    g.raff = v.raff;
    g.rstep = v.rstep;
  }
}

inline unsigned blocks_for(int64_t n, int threads = 256) {
  int64_t g = (n + threads - 1) / threads;
  return static_cast<unsigned>(g < 1 ? 1 : g);
}

int bits_for(uint64_t maxval) {
  int b = 0;
  while (b < 64 && (maxval >> b) != 0) ++b;
  return b;
}

// RAII list of device allocations released at scope exit.
struct DevPool {
  std::vector<void *> ptrs;
  ~DevPool() {
    for (void *p : ptrs) (void)hipFree(p);
  }
  template <typename T>
  qlt_status alloc(T **p, int64_t count) {
    *p = nullptr;
    if (count <= 0) count = 1;
    hipError_t e = hipMalloc(reinterpret_cast<void **>(p), sizeof(T) * static_cast<size_t>(count));
    if (e != hipSuccess) return hip_fail(e, "hipMalloc (plan scratch)", __FILE__, __LINE__);
    ptrs.push_back(*p);
    return QLT_OK;
  }
};

// Byte offsets of consecutive arrays in one allocation.
struct Packer {
  size_t bytes = 0;
  size_t add(size_t n) {
    const size_t at = bytes;
    bytes = (bytes + n + 255) & ~size_t(255);
    return at;
  }
};

// What the host keeps of a plan while it builds the work list.
struct HostBuild {
  std::vector<BlkShape> a, b;         // permuted view of every block
  std::vector<Tile> tiles;
  std::vector<ReduceItem> red;
  std::vector<PanelTile> ptiles;
  std::vector<PanelOut> pouts;
  std::vector<PanelTerm> pterms;
};

// Row panels on (1) or off (0) for plans built from now on (qlt_set_row_panels).
std::atomic<int> g_row_panels{1};

// Host form of split_offset (plain division).
int64_t host_split_offset(int64_t x, const int32_t *dims, const int32_t *strides, int n) {
  int64_t off = 0;
  for (int j = n - 1; j >= 0; --j) {
    const int64_t q = x / dims[j];
    off += (x - q * dims[j]) * strides[j];
    x = q;
  }
  return off;
}

// Row panels of the n <= 4 row class (PanelTile).  The output blocks are in
// ascending block order with A's saved axes leading, so the blocks sharing
// their coordinates on those axes are consecutive.  Each run of such blocks
// whose n <= 4 members together touch at most kPanelCols A' columns, with at
// most kPanelMaxOuts output columns and kPanelMaxTerms terms, becomes one
// panel; in_panel[o] marks its output blocks, which leave the row class.
qlt_status build_panels(qlt_plan *plan, HostBuild &hb, std::vector<char> &in_panel) {
  const int64_t n_c = plan->n_segs;
  in_panel.assign(static_cast<size_t>(n_c), 0);
  const int nr = plan->layout.a_nr;
  if (n_c == 0 || nr < 1 || nr > kPanelRowAxes || plan->c_rank < nr || plan->c_coords.empty()) return QLT_OK;
  if (plan->cls_tiles[kTileRows4] == 0) return QLT_OK;
  const auto &segs = plan->h_segs;
  const auto &ex = plan->h_exec;
  const int32_t cr = plan->c_rank;
  const GatherLayout &L = plan->layout;
  std::vector<PanelTile> &tiles = hb.ptiles;
  std::vector<PanelOut> &outs = hb.pouts;
  std::vector<PanelTerm> &terms = hb.pterms;
  // an A' column: (block, contracted index), and the block's element offset
  struct Col {
    int32_t blk, p;
    int64_t off;
    bool operator<(const Col &o) const { return blk != o.blk ? blk < o.blk : p < o.p; }
    bool operator==(const Col &o) const { return blk == o.blk && p == o.p; }
  };
  std::vector<Col> cols;
  std::vector<int64_t> members;
  int64_t o0 = 0;
  while (o0 < n_c) {
    // the run of output blocks with the coordinates of block o0 on A's saved axes
    int64_t o1 = o0 + 1;
    auto same_rows = [&](int64_t a, int64_t b) {
      for (int j = 0; j < nr; ++j)
        if (plan->c_coords[a * cr + j] != plan->c_coords[b * cr + j]) return false;
      return true;
    };
    while (o1 < n_c && same_rows(o0, o1)) ++o1;
    // its n <= 4 blocks, their A' columns in ascending order, and per output
    // column the terms in (task, k) order, which must be ascending in the
    // column.  The run's records are dropped again when it turns out not to
    // be a panel.
    cols.clear();
    members.clear();
    const size_t outs0 = outs.size(), terms0 = terms.size();
    bool ok = true;
    int32_t m = -1;
    // a column already in `cols` costs nothing: a run with more than
    // kPanelCols of them is no panel
    auto add_col = [&](const Col &c) {
      for (const Col &x : cols)
        if (x == c) return true;
      cols.push_back(c);
      return cols.size() <= static_cast<size_t>(kPanelCols);
    };
    for (int64_t o = o0; o < o1 && ok; ++o) {
      const Seg &sg = segs[static_cast<size_t>(o)];
      if (sg.cls != kTileRows4) continue;
      if (m >= 0 && sg.m != m) ok = false;
      m = sg.m;
      members.push_back(o);
      for (int32_t t = sg.t0; t < sg.t1 && ok; ++t) {
        const ExecTask &e = ex[static_cast<size_t>(t)];
        for (int32_t p = 0; p < e.k && ok; ++p) ok = add_col(Col{e.a_blk, p, e.a_off});
      }
    }
    ok = ok && !members.empty() && m > 0;
    if (ok) std::sort(cols.begin(), cols.end());
    for (size_t mi = 0; mi < members.size() && ok; ++mi) {
      const Seg &sg = segs[static_cast<size_t>(members[mi])];
      for (int32_t j = 0; j < sg.n && ok; ++j) {
        PanelOut po{static_cast<int32_t>(members[mi]), j, static_cast<int32_t>(terms.size() - terms0), 0};
        int32_t last = -1;
        for (int32_t t = sg.t0; t < sg.t1 && ok; ++t) {
          const ExecTask &e = ex[static_cast<size_t>(t)];
          const BlkShape &gB = hb.b[static_cast<size_t>(e.b_blk)];
          const int64_t bcol = host_split_offset(j, gB.cdim, gB.cstr, L.b_nc);
          for (int32_t p = 0; p < e.k && ok; ++p) {
            int32_t c = 0;
            while (!(cols[static_cast<size_t>(c)].blk == e.a_blk && cols[static_cast<size_t>(c)].p == p)) ++c;
            if (c <= last) {
              ok = false;
              break;
            }
            last = c;
            po.mask |= 1 << c;
            const int64_t brow = host_split_offset(p, gB.rdim, gB.rstr, L.b_nr);
            terms.push_back(PanelTerm{e.b_off + brow + bcol, c, 0});
          }
        }
        outs.push_back(po);
        ok = ok && outs.size() - outs0 <= static_cast<size_t>(kPanelMaxOuts) &&
             terms.size() - terms0 <= static_cast<size_t>(kPanelMaxTerms);
      }
    }
    if (!ok) {
      outs.resize(outs0);
      terms.resize(terms0);
    } else {
      PanelTile pt{};
      const BlkShape &g0 = hb.a[static_cast<size_t>(cols[0].blk)];
      for (int l = 0; l < kPanelRowAxes; ++l) {
        pt.rdim[l] = l < nr ? g0.rdim[l] : 1;
        magic_of(static_cast<uint32_t>(pt.rdim[l]), pt.rmag[l], pt.rsh[l]);
      }
      for (size_t c = 0; c < cols.size(); ++c) {
        const BlkShape &g = hb.a[static_cast<size_t>(cols[c].blk)];
        pt.cbase[c] = cols[c].off + host_split_offset(cols[c].p, g.cdim, g.cstr, L.a_nc);
        for (int l = 0; l < nr; ++l) pt.cstr[c][l] = g.rstr[l];
      }
      pt.pair1 = 0;
      for (int c = 0; c + 1 < static_cast<int>(cols.size()) && pt.pair1 == 0; ++c) {
        bool adj = pt.cbase[c + 1] == pt.cbase[c] + 1;
        for (int l = 0; l < kPanelRowAxes; ++l) adj = adj && pt.cstr[c][l] == pt.cstr[c + 1][l];
        if (adj) pt.pair1 = c + 1;
      }
      pt.m = m;
      pt.n_cols = static_cast<int32_t>(cols.size());
      pt.n_outs = static_cast<int32_t>(outs.size() - outs0);
      pt.n_terms = static_cast<int32_t>(terms.size() - terms0);
      pt.out0 = static_cast<int32_t>(outs0);
      pt.term0 = static_cast<int32_t>(terms0);
      for (int32_t r0 = 0; r0 < m; r0 += kPanelRows) {
        pt.r0 = r0;
        tiles.push_back(pt);
      }
      for (int64_t o : members) {
        in_panel[static_cast<size_t>(o)] = 1;
        const Seg &sg = segs[static_cast<size_t>(o)];
        for (int32_t t = sg.t0; t < sg.t1; ++t)
          plan->panel_mkn += static_cast<double>(sg.m) * static_cast<double>(ex[static_cast<size_t>(t)].k) * sg.n;
        plan->panel_elems += static_cast<double>(sg.m) * sg.n;
      }
      plan->panel_elems += static_cast<double>(m) * static_cast<double>(cols.size());
    }
    o0 = o1;
  }
  QLT_CHECK_ARG(static_cast<int64_t>(terms.size()) < (int64_t(1) << 31) &&
                    static_cast<int64_t>(tiles.size()) < (int64_t(1) << 31),
                "qlt_plan_build: too many row panels");
  plan->n_ptiles = static_cast<int64_t>(tiles.size());
  if (tiles.empty()) return QLT_OK;
  // what the row class keeps
  plan->cls_mkn[kTileRows4] = 0.0;
  plan->cls_elems[kTileRows4] = 0.0;
  std::vector<char> seen_a(static_cast<size_t>(plan->n_a_blks), 0), seen_b(static_cast<size_t>(plan->n_b_blks), 0);
  for (int64_t o = 0; o < n_c; ++o) {
    const Seg &sg = segs[static_cast<size_t>(o)];
    if (sg.cls != kTileRows4 || in_panel[static_cast<size_t>(o)]) continue;
    plan->cls_mkn[kTileRows4] += static_cast<double>(sg.m) * sg.n * static_cast<double>(sg.k_total);
    plan->cls_elems[kTileRows4] += static_cast<double>(sg.m) * sg.n;
    for (int32_t t = sg.t0; t < sg.t1; ++t) {
      const ExecTask &e = ex[static_cast<size_t>(t)];
      if (!seen_a[e.a_blk]) {
        seen_a[e.a_blk] = 1;
        plan->cls_elems[kTileRows4] += static_cast<double>(sg.m) * e.k;
      }
      if (!seen_b[e.b_blk]) {
        seen_b[e.b_blk] = 1;
        plan->cls_elems[kTileRows4] += static_cast<double>(e.k) * sg.n;
      }
    }
  }
  return QLT_OK;
}

// Beyond kPanelCols, so that what a row panel may take stays with the row class.
constexpr int64_t kRows4MaxK = 64;

// Class of every n <= 16 output block, from measurements of single blocks of m
// rows in FP64, complex128 and complex64 with A in either memory order, and of
// blocks of many short tasks (us; k: contracted extent).
//   4 < n <= 16: a chain of steps shared by four waves (kTileNarrow) while the
// 32-row tiles are too few to fill the chip, else a tile per wave
// (kTileNarrowRows): shared, waves without a step idle and all four meet in LDS.
// The line is 1024 tiles for each 16-k step, 2048 for each of more than four that
// are not short (shared | a wave each, n = 8, complex128: k = 16, m = 10^4 5.0 | 6.5, m =
// 10^5 17.8 | 13.2, m = 10^6 163 | 96; k = 64, m = 10^5 29.9 | 31.4; k = 128, m = 3 10^5
// 150 | 157, m = 10^6 474 | 458; complex64, k = 16, m = 10^6 150 | 69).
//   n <= 4, k <= 64: the row class, in which row panels look for their members.
//   n <= 4, k > 64: the row class walks its steps one after the other (a U(1)
// chi = 16 pair of rank-4 tensors, FP64: 43 us, as kTileNarrow 13), but reads A
// once in whole lines when k is not A's innermost axis or the tasks are short,
// and is the faster one when its 1024-row tiles are many (n = 1, rows | kTileNarrow:
// k = 128, k not innermost, complex64, m = 10^5 43 | 43, m = 10^6 181 | 391; k
// innermost, FP64, m = 10^6 1089 | 223; 100 tasks of k = 1, FP64, m = 3000 25 | 14,
// m = 30 000 32 | 46, m = 10^5 43 | 127; 40 tasks of k = 4, m = 30 000 28 | 24).
constexpr int64_t kShortK = 4;
constexpr int64_t kNarrowTilesPerStep = 1024;
constexpr int64_t kRowsTilesStream = 256;   // tiles
constexpr int64_t kRowsStepsShort = 1536;   // tiles times steps
void choose_narrow_classes(qlt_plan *plan, const std::vector<BlkShape> &a) {
  const int64_t rows4 = plan->cls_tiles[kTileRows4], tiles32 = plan->cls_tiles[kTileNarrow];
  for (Seg &sg : plan->h_segs) {
    const bool long_rows = sg.cls == kTileRows4 && sg.k_total > kRows4MaxK;
    const bool many_tiles = sg.cls == kTileNarrow && tiles32 >= kNarrowTilesPerStep;
    if (!long_rows && !many_tiles) continue;
    int64_t steps = 0;
    bool all_short = true, streams = true;   // streams: no longer task has k innermost in A
    for (int32_t t = sg.t0; t < sg.t1; ++t) {
      const ExecTask &e = plan->h_exec[static_cast<size_t>(t)];
      const BlkShape &ga = a[static_cast<size_t>(e.a_blk)];
      steps += chunks_from(0, e.k);
      if (e.k > kShortK) {
        all_short = false;
        if (ga.plain || ga.fastcol) streams = false;
      }
    }
    int32_t to = sg.cls;
    if (long_rows) {
      const bool rows = (all_short && rows4 * steps >= kRowsStepsShort) || (streams && rows4 >= kRowsTilesStream);
      if (!rows) to = kTileNarrow;
    } else if (tiles32 >= kNarrowTilesPerStep * steps * (steps > 4 && !all_short ? 2 : 1)) {
      to = kTileNarrowRows;
    }
    if (to == sg.cls) continue;
    plan->cls_tiles[sg.cls] -= tiles_of(sg.cls, sg.m, sg.n);
    sg.cls = to;
    plan->cls_tiles[sg.cls] += tiles_of(sg.cls, sg.m, sg.n);
  }
}

// k-slicing of long tiles (MFMA and row classes alike).  Per class, a step budget Q = max(kMinSliceChunks,
// ceil(total steps / T)) is set, T = kSliceTargetWGsMfma (MFMA classes) or kSliceTargetWGs (row classes)
// unless tuned (qlt_tuning); a tile of w > Q steps is cut into
// ceil(w / Q) (at most kMaxSlices) slices of nearly equal length along its
// (task, k-chunk) sequence, each writing an unscaled partial sum that a
// reduction kernel adds in slice order.  Classes whose tiles are many and even
// stay unsliced; few or long tiles (a contraction over a long k onto a small
// output) spread over the chip.  Slices of >= kMinSliceChunks steps keep the
// partial-sum traffic small against the slice's MFMA work.
constexpr int64_t kSliceTargetWGs = 2048;
// The MFMA classes aim lower: fewer, longer slices (and less partial-sum
// traffic) measured faster on every matvec chain here than 2048.
constexpr int64_t kSliceTargetWGsMfma = 512;
constexpr int64_t kMinSliceChunks = 8;
// The n <= 16 class spreads a tile's chunks over four waves by itself: slices
// as short as the MFMA classes' would leave two chunks to a wave.
constexpr int64_t kMinSliceChunksNarrow = 32;
constexpr int64_t kMaxSlices = 64;

// Tiles of every output block, class by class: MFMA tiles longest first, row
// tiles by the A block they start on; long ones cut into k-slices.
qlt_status build_tiles(qlt_plan *plan, HostBuild &hb) {
  const auto &segs = plan->h_segs;
  const auto &ex = plan->h_exec;
  auto steps_of = [](int64_t k) { return (k + kKChunk - 1) / kKChunk; };
  std::vector<int64_t> seg_steps(segs.size(), 0);
  std::vector<int32_t> by_cls[kNumTileClasses];
  std::vector<char> in_panel;
  if (plan->panels_enabled) QLT_TRY(build_panels(plan, hb, in_panel));
  for (size_t o = 0; o < segs.size(); ++o) {
    if (!in_panel.empty() && in_panel[o]) continue;   // runs as a row panel
    for (int32_t t = segs[o].t0; t < segs[o].t1; ++t) seg_steps[o] += steps_of(ex[static_cast<size_t>(t)].k);
    by_cls[segs[o].cls].push_back(static_cast<int32_t>(o));
  }
  std::vector<Tile> cl;
  int64_t part_doubles = 0;
  for (int32_t cls = 0; cls < kNumTileClasses; ++cls) {
    // partial-sum doubles of one slice (complex), in the kernels' thread order
    const int64_t slice_doubles = is_mfma_class(cls) ? int64_t(mfma_tile_m(cls)) * mfma_tile_n(cls) * 2
                                                     : int64_t(rows_per_tile(cls)) * (cls == kTileRows4 ? 4 : 16) * 2;
    int64_t total = 0, count = 0;
    for (int32_t o : by_cls[cls]) {
      const int64_t n = tiles_of(cls, segs[static_cast<size_t>(o)].m, segs[static_cast<size_t>(o)].n);
      total += n * seg_steps[static_cast<size_t>(o)];
      count += n;
    }
    // tuned workgroup target of the class (qlt_tuning; -1: unsliced)
    const bool unsliced = plan->slice_target[cls] < 0;
    const int64_t target = plan->slice_target[cls] > 0 ? plan->slice_target[cls]
                                                       : (is_mfma_class(cls) ? kSliceTargetWGsMfma : kSliceTargetWGs);
    const int64_t q =
        std::max(cls == kTileNarrow ? kMinSliceChunksNarrow : kMinSliceChunks, (total + target - 1) / target);
    cl.clear();
    cl.reserve(static_cast<size_t>(count));
    int64_t parts = 0;
    const size_t red0 = hb.red.size();
    for (int32_t o : by_cls[cls]) {
      const Seg &s = segs[static_cast<size_t>(o)];
      const int64_t w = seg_steps[static_cast<size_t>(o)];
      const int64_t ns = unsliced ? 1 : std::min(kMaxSlices, (w + q - 1) / q);
      const int64_t n = tiles_of(cls, s.m, s.n);
      const int32_t ntn = is_mfma_class(cls) ? (s.n + mfma_tile_n(cls) - 1) / mfma_tile_n(cls) : 1;
      for (int64_t i = 0; i < n; ++i) {
        const Tile t{o, static_cast<int32_t>(i / ntn), static_cast<int32_t>(i % ntn), cls, s.t0, 0,
                     static_cast<int32_t>(w), -1};
        if (ns <= 1) {
          cl.push_back(t);
          continue;
        }
        hb.red.push_back(ReduceItem{o, t.tm, t.tn, cls, static_cast<int32_t>(parts), static_cast<int32_t>(ns)});
        int32_t task = s.t0;
        int64_t in_task = 0;     // steps already taken inside `task`
        for (int64_t sl = 0; sl < ns; ++sl) {
          const int64_t len = w / ns + (sl < w % ns ? 1 : 0);
          Tile u = t;
          u.t_begin = task;
          u.k_begin = static_cast<int32_t>(in_task * kKChunk);
          u.n_chunks = static_cast<int32_t>(len);
          u.part = static_cast<int32_t>(parts + sl);
          cl.push_back(u);
          for (int64_t rem = len; rem > 0;) {
            const int64_t left = steps_of(ex[static_cast<size_t>(task)].k) - in_task;
            if (rem < left) {
              in_task += rem;
              rem = 0;
            } else {
              rem -= left;
              ++task;
              in_task = 0;
            }
          }
        }
        parts += ns;
      }
    }
    if (is_mfma_class(cls)) {
      std::stable_sort(cl.begin(), cl.end(), [](const Tile &a, const Tile &b) { return a.n_chunks > b.n_chunks; });
    } else {
      // row tiles are short and bound by reading A: tiles that start on the
      // same A block rows run next to each other (and on one XCD), so the
      // output blocks that re-read an A block find it in L2
      std::stable_sort(cl.begin(), cl.end(), [&](const Tile &a, const Tile &b) {
        const int32_t ka = ex[static_cast<size_t>(a.t_begin)].a_blk, kb = ex[static_cast<size_t>(b.t_begin)].a_blk;
        return ka != kb ? ka < kb : a.tm < b.tm;
      });
    }
    hb.tiles.insert(hb.tiles.end(), cl.begin(), cl.end());
    plan->cls_tiles[cls] = static_cast<int64_t>(cl.size());
    plan->cls_red[cls] = static_cast<int64_t>(hb.red.size() - red0);
    // every class gets its own region: the class kernels run concurrently
    plan->cls_part_off[cls] = part_doubles;
    part_doubles += parts * slice_doubles;
  }
  QLT_CHECK_ARG(static_cast<int64_t>(hb.tiles.size()) < (int64_t(1) << 31),
                "qlt_plan_build: too many tiles after k-slicing");
  plan->n_tiles = static_cast<int64_t>(hb.tiles.size());
  plan->part_doubles = hb.red.empty() ? 0 : static_cast<size_t>(part_doubles);
  return QLT_OK;
}

qlt_status validate_desc(const qlt_bsdt_desc *d, const char *name) {
  const std::string n(name);
  QLT_CHECK_ARG(d != nullptr, "qlt_plan_build: null descriptor " + n);
  QLT_CHECK_ARG(d->rank >= 1 && d->rank <= QLT_MAX_RANK,
                "qlt_plan_build: rank of " + n + " must be in 1.." + std::to_string(QLT_MAX_RANK));
  QLT_CHECK_ARG(d->n_blks >= 0 && d->n_blks < (int64_t(1) << 31),
                "qlt_plan_build: bad block count of " + n);
  if (d->n_blks == 0) return QLT_OK;
  QLT_CHECK_ARG(d->blk_shape && d->blk_coords && d->blk_dims && d->blk_offsets,
                "qlt_plan_build: null array in descriptor " + n);
  for (int j = 0; j < d->rank; ++j)
    QLT_CHECK_ARG(d->blk_shape[j] >= 1 && d->blk_shape[j] < (int64_t(1) << 31),
                  "qlt_plan_build: bad sector count in " + n);
  uint64_t prev_idx = 0;
  for (int64_t i = 0; i < d->n_blks; ++i) {
    uint64_t idx = 0;
    int64_t size = 1;
    for (int j = 0; j < d->rank; ++j) {
      const int64_t c = d->blk_coords[i * d->rank + j];
      const int64_t dim = d->blk_dims[i * d->rank + j];
      QLT_CHECK_ARG(c >= 0 && c < d->blk_shape[j], "qlt_plan_build: block coordinate out of range in " + n);
      QLT_CHECK_ARG(dim >= 1 && dim < (int64_t(1) << 31), "qlt_plan_build: bad block dimension in " + n);
      idx = idx * static_cast<uint64_t>(d->blk_shape[j]) + static_cast<uint64_t>(c);
      size *= dim;
      QLT_CHECK_ARG(size < (int64_t(1) << 31), "qlt_plan_build: block of " + n + " exceeds 2^31 elements");
    }
    QLT_CHECK_ARG(i == 0 || idx > prev_idx,
                  "qlt_plan_build: blocks of " + n + " must be in strictly ascending block index");
    QLT_CHECK_ARG(d->blk_offsets[i] >= 0, "qlt_plan_build: negative block offset in " + n);
    prev_idx = idx;
  }
  return QLT_OK;
}

}  // namespace


namespace {

// Block index of every block of a descriptor (row-major over blk_shape).
std::vector<int64_t> block_indices(const qlt_bsdt_desc *d) {
  std::vector<int64_t> idx(d->n_blks);
  for (int64_t i = 0; i < d->n_blks; ++i) {
    uint64_t v = 0;
    for (int j = 0; j < d->rank; ++j)
      v = v * static_cast<uint64_t>(d->blk_shape[j]) + static_cast<uint64_t>(d->blk_coords[i * d->rank + j]);
    idx[i] = static_cast<int64_t>(v);
  }
  return idx;
}

qlt_status check_axes(const qlt_bsdt_desc *a, const qlt_bsdt_desc *b, int32_t n_ctrct,
                      const int32_t *a_ctrct_axes, const int32_t *b_ctrct_axes, int32_t n_a_saved,
                      const int32_t *a_saved_axes, int32_t n_b_saved, const int32_t *b_saved_axes) {
  QLT_CHECK_ARG(n_ctrct >= 0 && n_a_saved >= 0 && n_b_saved >= 0, "qlt_plan_build: negative axis count");
  QLT_CHECK_ARG(n_ctrct + n_a_saved == a->rank, "qlt_plan_build: A axes do not cover A's rank");
  QLT_CHECK_ARG(n_ctrct + n_b_saved == b->rank, "qlt_plan_build: B axes do not cover B's rank");
  QLT_CHECK_ARG(n_ctrct == 0 || (a_ctrct_axes && b_ctrct_axes), "qlt_plan_build: null contracted axes");
  QLT_CHECK_ARG(n_a_saved == 0 || a_saved_axes, "qlt_plan_build: null A saved axes");
  QLT_CHECK_ARG(n_b_saved == 0 || b_saved_axes, "qlt_plan_build: null B saved axes");
  QLT_CHECK_ARG(n_a_saved + n_b_saved <= QLT_MAX_RANK, "qlt_plan_build: output rank exceeds QLT_MAX_RANK");
  std::vector<int> seen_a(a->rank, 0), seen_b(b->rank, 0);
  for (int j = 0; j < n_ctrct; ++j) {
    QLT_CHECK_ARG(a_ctrct_axes[j] >= 0 && a_ctrct_axes[j] < a->rank, "qlt_plan_build: bad A axis");
    QLT_CHECK_ARG(b_ctrct_axes[j] >= 0 && b_ctrct_axes[j] < b->rank, "qlt_plan_build: bad B axis");
    seen_a[a_ctrct_axes[j]]++;
    seen_b[b_ctrct_axes[j]]++;
  }
  for (int j = 0; j < n_a_saved; ++j) {
    QLT_CHECK_ARG(a_saved_axes[j] >= 0 && a_saved_axes[j] < a->rank, "qlt_plan_build: bad A saved axis");
    seen_a[a_saved_axes[j]]++;
  }
  for (int j = 0; j < n_b_saved; ++j) {
    QLT_CHECK_ARG(b_saved_axes[j] >= 0 && b_saved_axes[j] < b->rank, "qlt_plan_build: bad B saved axis");
    seen_b[b_saved_axes[j]]++;
  }
  for (int v : seen_a) QLT_CHECK_ARG(v == 1, "qlt_plan_build: A axes are not a permutation of A's axes");
  for (int v : seen_b) QLT_CHECK_ARG(v == 1, "qlt_plan_build: B axes are not a permutation of B's axes");
  if (a->n_blks > 0 && b->n_blks > 0)
    for (int j = 0; j < n_ctrct; ++j)
      QLT_CHECK_ARG(a->blk_shape[a_ctrct_axes[j]] == b->blk_shape[b_ctrct_axes[j]],
                    "qlt_plan_build: contracted indexes have different sector counts");
  return QLT_OK;
}

}  // namespace

extern "C" {

qlt_status qlt_plan_build(const qlt_bsdt_desc *a, const qlt_bsdt_desc *b, int32_t n_ctrct,
                          const int32_t *a_ctrct_axes, const int32_t *b_ctrct_axes,
                          int32_t n_a_saved, const int32_t *a_saved_axes, int32_t n_b_saved,
                          const int32_t *b_saved_axes, void *stream, qlt_plan **plan_out) {
  QLT_REQUIRE_INIT();
  QLT_CHECK_ARG(plan_out != nullptr, "qlt_plan_build: null output");
  *plan_out = nullptr;
  QLT_TRY(validate_desc(a, "A"));
  QLT_TRY(validate_desc(b, "B"));
  QLT_TRY(check_axes(a, b, n_ctrct, a_ctrct_axes, b_ctrct_axes, n_a_saved, a_saved_axes, n_b_saved,
                     b_saved_axes));
  hipStream_t st = as_stream(stream);
  QLT_CHECK_ARG(!stream_capturing(st), "qlt_plan_build: cannot build a plan under graph capture");
  const int32_t c_rank = n_a_saved + n_b_saved;

  PlanArgs args{};
  args.a_rank = a->rank;
  args.b_rank = b->rank;
  args.n_ctrct = n_ctrct;
  args.n_a_saved = n_a_saved;
  args.n_b_saved = n_b_saved;
  args.c_rank = c_rank;
  for (int j = 0; j < n_ctrct; ++j) {
    args.a_ctrct[j] = a_ctrct_axes[j];
    args.b_ctrct[j] = b_ctrct_axes[j];
  }
  for (int j = 0; j < n_a_saved; ++j) args.a_saved[j] = a_saved_axes[j];
  for (int j = 0; j < n_b_saved; ++j) args.b_saved[j] = b_saved_axes[j];
  args.c_is_scalar = (c_rank == 0) ? 1 : 0;
  const qlt_tuning tun = tuning_snapshot();
  std::memcpy(args.cls_table, tun.tile_class, sizeof(args.cls_table));

  auto plan = std::make_unique<qlt_plan>();
  plan->device = current_device();
  plan->c_rank = c_rank;
  plan->c_is_scalar = args.c_is_scalar;
  for (int c = 0; c < kNumTileClasses; ++c) plan->slice_target[c] = tun.slice_target[tuning_class(c)];
  plan->n_a_blks = a->n_blks;
  plan->n_b_blks = b->n_blks;
  {
    GatherLayout &L = plan->layout;
    L.a_nr = n_a_saved;
    L.a_nc = n_ctrct;
    L.b_nr = n_ctrct;
    L.b_nc = n_b_saved;
    L.a_kfast = (n_ctrct > 0 && a_ctrct_axes[n_ctrct - 1] == a->rank - 1) ? 1 : 0;
    L.b_nfast = (n_b_saved > 0 && b_saved_axes[n_b_saved - 1] == b->rank - 1) ? 1 : 0;
  }
  const int64_t na = a->n_blks, nb = b->n_blks;
  for (int64_t i = 0; i < na; ++i) {
    int64_t sz = 1;
    for (int j = 0; j < a->rank; ++j) sz *= a->blk_dims[i * a->rank + j];
    plan->max_blk_elems_a = std::max(plan->max_blk_elems_a, sz);
    plan->a_raw_extent = std::max(plan->a_raw_extent, a->blk_offsets[i] + sz);
  }
  for (int64_t i = 0; i < nb; ++i) {
    int64_t sz = 1;
    for (int j = 0; j < b->rank; ++j) sz *= b->blk_dims[i * b->rank + j];
    plan->max_blk_elems_b = std::max(plan->max_blk_elems_b, sz);
    plan->b_raw_extent = std::max(plan->b_raw_extent, b->blk_offsets[i] + sz);
  }
  if (na == 0 || nb == 0) {
    *plan_out = plan.release();
    return QLT_OK;
  }

  // Output block strides, row-major over the output sector counts.
  uint64_t c_space = 1;
  {
    std::vector<int64_t> cshape;
    for (int j = 0; j < n_a_saved; ++j) cshape.push_back(a->blk_shape[a_saved_axes[j]]);
    for (int j = 0; j < n_b_saved; ++j) cshape.push_back(b->blk_shape[b_saved_axes[j]]);
    unsigned __int128 s = 1;
    for (int j = c_rank - 1; j >= 0; --j) {
      args.c_stride[j] = static_cast<int64_t>(s);
      s *= static_cast<uint64_t>(cshape[j]);
      QLT_CHECK_ARG(s < (static_cast<unsigned __int128>(1) << 63),
                    "qlt_plan_build: output block index space exceeds 2^63");
    }
    c_space = static_cast<uint64_t>(s);
  }

  // ---- block metadata to the device, in one copy ----
  Packer up;
  const size_t o_ac = up.add(4 * na * a->rank), o_ad = up.add(4 * na * a->rank);
  const size_t o_bc = up.add(4 * nb * b->rank), o_bd = up.add(4 * nb * b->rank);
  const size_t up_bytes = up.bytes;
  const size_t o_hash = up.add(8 * (na + nb)), o_cnt = up.add(8 * na), o_start = up.add(8 * na), o_nt = up.add(8);
  DevPool pool;
  char *d0 = nullptr;
  QLT_TRY(pool.alloc(&d0, static_cast<int64_t>(up.bytes)));
  PinnedStaging stage(st);
  QLT_TRY(stage.reserve(up_bytes));
  int32_t *const h_ac = stage.at<int32_t>(o_ac), *const h_ad = stage.at<int32_t>(o_ad);
  int32_t *const h_bc = stage.at<int32_t>(o_bc), *const h_bd = stage.at<int32_t>(o_bd);
  for (int64_t i = 0; i < na * a->rank; ++i) {
    h_ac[i] = static_cast<int32_t>(a->blk_coords[i]);
    h_ad[i] = static_cast<int32_t>(a->blk_dims[i]);
  }
  for (int64_t i = 0; i < nb * b->rank; ++i) {
    h_bc[i] = static_cast<int32_t>(b->blk_coords[i]);
    h_bd[i] = static_cast<int32_t>(b->blk_dims[i]);
  }
  auto dev = [&](size_t off) { return static_cast<void *>(d0 + off); };
  const auto *d_ac = static_cast<const int32_t *>(dev(o_ac)), *d_ad = static_cast<const int32_t *>(dev(o_ad));
  const auto *d_bc = static_cast<const int32_t *>(dev(o_bc)), *d_bd = static_cast<const int32_t *>(dev(o_bd));
  auto *d_ha = static_cast<uint64_t *>(dev(o_hash)), *d_hb = d_ha + na;
  auto *d_cnt = static_cast<int64_t *>(dev(o_cnt)), *d_start = static_cast<int64_t *>(dev(o_start));
  auto *d_nt = static_cast<int64_t *>(dev(o_nt));
  QLT_HIP(hipMemcpyAsync(d0, stage.at<char>(0), up_bytes, hipMemcpyHostToDevice, st));

  // ---- 1. part hashes; 2. matches per A block and task slots ----
  hipLaunchKernelGGL(k_part_hash, dim3(blocks_for(na + nb)), dim3(256), 0, st, d_ac, na, d_bc, nb, args, d_ha);
  hipLaunchKernelGGL(k_count, dim3(blocks_for(na)), dim3(256), 0, st, d_ha, na, d_hb, nb,
                     args.c_is_scalar, d_cnt);
  hipLaunchKernelGGL(k_scan_excl, dim3(1), dim3(1024), 0, st, d_cnt, d_start, na, d_nt);
  QLT_HIP(hipGetLastError());
  PinnedStaging back(st);
  QLT_TRY(back.reserve(8));
  QLT_HIP(hipMemcpyAsync(back.at<char>(0), d_nt, 8, hipMemcpyDeviceToHost, st));
  // meanwhile: the permuted view of every block
  HostBuild hb;
  hb.a.resize(static_cast<size_t>(na));
  hb.b.resize(static_cast<size_t>(nb));
  for (int64_t i = 0; i < na; ++i)
    blk_shape(h_ad + i * a->rank, a->rank, args.a_saved, n_a_saved, args.a_ctrct, n_ctrct, hb.a[static_cast<size_t>(i)]);
  for (int64_t i = 0; i < nb; ++i)
    blk_shape(h_bd + i * b->rank, b->rank, args.b_ctrct, n_ctrct, args.b_saved, n_b_saved, hb.b[static_cast<size_t>(i)]);
  const std::vector<int64_t> h_aidx = block_indices(a), h_bidx = block_indices(b);
  QLT_HIP(hipStreamSynchronize(st));
  const int64_t nt = *back.at<int64_t>(0);
  if (nt == 0) {
    *plan_out = plan.release();
    return QLT_OK;
  }
  QLT_CHECK_ARG(nt < (int64_t(1) << 31), "qlt_plan_build: more than 2^31 tasks");

  // ---- 2. tasks, and their stable sort by output block index ----
  Packer tp;
  const bool by_rank = nt <= kRankMaxTasks;
  const size_t o_task = tp.add(8 * nt), o_k0 = tp.add(8 * nt), o_v0 = tp.add(4 * nt), o_k1 = tp.add(8 * nt),
               o_v1 = tp.add(4 * nt), o_rank = tp.add(4 * nt);
  char *d1 = nullptr;
  QLT_TRY(pool.alloc(&d1, static_cast<int64_t>(tp.bytes)));
  auto *d_tasks = reinterpret_cast<DevTask *>(d1 + o_task);
  auto *d_k0 = reinterpret_cast<uint64_t *>(d1 + o_k0), *d_k1 = reinterpret_cast<uint64_t *>(d1 + o_k1);
  auto *d_v0 = reinterpret_cast<int32_t *>(d1 + o_v0), *d_v1 = reinterpret_cast<int32_t *>(d1 + o_v1);
  auto *d_rank = reinterpret_cast<int32_t *>(d1 + o_rank);
  hipLaunchKernelGGL(k_emit, dim3(blocks_for(na * 64)), dim3(256), 0, st, d_ha, na, d_hb, nb, d_start, d_ac, d_bc, args,
                     d_tasks, d_k0, d_v0, d_rank);
  const int passes = (bits_for(c_space - 1) + 7) / 8;
  bool in_k1 = true;
  if (by_rank) {
    hipLaunchKernelGGL(k_rank, dim3(blocks_for(nt), static_cast<unsigned>((nt + kRankChunk - 1) / kRankChunk)),
                       dim3(256), 0, st, d_k0, nt, d_rank);
    hipLaunchKernelGGL(k_place, dim3(blocks_for(nt)), dim3(256), 0, st, d_k0, d_rank, nt, d_k1, d_v1);
  } else {
    if (passes > 0)
      hipLaunchKernelGGL(k_radix_sort, dim3(1), dim3(1024), 0, st, d_k0, d_v0, d_k1, d_v1, nt, passes);
    in_k1 = (passes & 1) != 0;
  }
  QLT_HIP(hipGetLastError());
  Packer bp;
  const size_t b_task = bp.add(8 * nt), b_sk = bp.add(8 * nt), b_sv = bp.add(4 * nt);
  QLT_TRY(back.reserve(bp.bytes));
  QLT_HIP(hipMemcpyAsync(back.at<char>(b_task), d_tasks, 8 * nt, hipMemcpyDeviceToHost, st));
  QLT_HIP(hipMemcpyAsync(back.at<char>(b_sk), in_k1 ? d_k1 : d_k0, 8 * nt, hipMemcpyDeviceToHost, st));
  QLT_HIP(hipMemcpyAsync(back.at<char>(b_sv), in_k1 ? d_v1 : d_v0, 4 * nt, hipMemcpyDeviceToHost, st));
  plan->tasks.resize(static_cast<size_t>(nt));
  plan->h_exec.resize(static_cast<size_t>(nt));
  QLT_HIP(hipStreamSynchronize(st));
  const DevTask *const h_task = back.at<DevTask>(b_task);
  const uint64_t *const h_sk = back.at<uint64_t>(b_sk);
  const int32_t *const h_sv = back.at<int32_t>(b_sv);

  // ---- 3 - 5. task records in execution order, output blocks (first touch
  // -> beta 0) and their offsets ----
  std::vector<Seg> &segs = plan->h_segs;
  {
    int64_t heads = 1;
    for (int64_t p = 1; p < nt; ++p) heads += h_sk[p] != h_sk[p - 1];
    const size_t n = static_cast<size_t>(heads);
    segs.reserve(n);
    if (!args.c_is_scalar) {
      plan->c_blk_idx.reserve(n);
      plan->c_offsets.reserve(n);
      plan->c_coords.reserve(n * static_cast<size_t>(c_rank));
      plan->c_dims.reserve(n * static_cast<size_t>(c_rank));
    }
  }
  int64_t c_raw = 0, kmax = 0, sum_mkn = 0, n_tiles = 0;
  for (int64_t p = 0; p < nt; ++p) {
    const int32_t g = h_sv[p];
    const DevTask dt = h_task[g];
    const BlkShape &sa = hb.a[static_cast<size_t>(dt.a_pos)], &sb = hb.b[static_cast<size_t>(dt.b_pos)];
    const bool head = p == 0 || h_sk[p] != h_sk[p - 1];
    const int64_t m = sa.nrows, k = sa.ncols, n = sb.ncols;
    if (head) {
      Seg sg{};
      sg.c_off = c_raw;
      sg.m = static_cast<int32_t>(m);
      sg.n = static_cast<int32_t>(n);
      sg.t0 = static_cast<int32_t>(p);
      sg.cls = tuned_tile_class(m, n, args.cls_table);
      sg.flags = kSegAPlain | kSegBPlain | kSegAColAffine | kSegBRowAffine;
      segs.push_back(sg);
      c_raw += m * n;
      plan->cls_tiles[sg.cls] += tiles_of(sg.cls, m, n);
      // The reference keeps no block for a rank-0 output; its raw size is 1.
      if (!args.c_is_scalar) {
        plan->c_blk_idx.push_back(static_cast<int64_t>(h_sk[p]));
        plan->c_offsets.push_back(sg.c_off);
        for (int j = 0; j < n_a_saved; ++j) {
          plan->c_coords.push_back(h_ac[int64_t(dt.a_pos) * a->rank + args.a_saved[j]]);
          plan->c_dims.push_back(sa.rdim[j]);
        }
        for (int j = 0; j < n_b_saved; ++j) {
          plan->c_coords.push_back(h_bc[int64_t(dt.b_pos) * b->rank + args.b_saved[j]]);
          plan->c_dims.push_back(sb.cdim[j]);
        }
      }
    }
    Seg &sg = segs.back();
    sg.t1 = static_cast<int32_t>(p + 1);
    sg.k_total += k;
    kmax = std::max(kmax, sg.k_total);
    sum_mkn += m * k * n;
    // the flags hold for every task of the block: plain blocks run without
    // divisions, blocks affine in k on per-element pointers
    if (!sa.plain) sg.flags &= ~kSegAPlain;
    if (!sb.plain) sg.flags &= ~kSegBPlain;
    if (!sa.plain && !sa.caff) sg.flags &= ~kSegAColAffine;
    if (!sb.plain && !sb.raff) sg.flags &= ~kSegBRowAffine;
    const int64_t a_off = a->blk_offsets[dt.a_pos], b_off = b->blk_offsets[dt.b_pos];
    plan->tasks[static_cast<size_t>(g)] =
        qlt_task{h_aidx[static_cast<size_t>(dt.a_pos)], a_off, h_bidx[static_cast<size_t>(dt.b_pos)], b_off,
                 static_cast<int64_t>(h_sk[p]), sg.c_off, m, k, n, 1.0, head ? 0.0 : 1.0};
    plan->h_exec[static_cast<size_t>(p)] =
        ExecTask{a_off, b_off, dt.a_pos, dt.b_pos, static_cast<int32_t>(k), 0};
  }
  const int64_t n_c = static_cast<int64_t>(segs.size());
  choose_narrow_classes(plan.get(), hb.a);
  n_tiles = 0;
  for (int c = 0; c < kNumTileClasses; ++c) n_tiles += plan->cls_tiles[c];
  QLT_CHECK_ARG(n_tiles < (int64_t(1) << 31), "qlt_plan_build: more than 2^31 output tiles");
  QLT_CHECK_ARG(kmax < (int64_t(1) << 40), "qlt_plan_build: contracted extent of an output block exceeds 2^40");
  plan->n_exec = nt;
  plan->n_segs = n_c;
  plan->c_raw_size = c_raw;
  plan->sum_mkn = sum_mkn;
  // Per-class algorithmic work (m*k*n summed) and compulsory elements
  // (distinct A and B blocks a class reads, plus the C blocks it writes).
  {
    std::vector<uint8_t> seen_a(static_cast<size_t>(na), 0), seen_b(static_cast<size_t>(nb), 0);
    for (const Seg &s : segs) {
      plan->cls_mkn[s.cls] += static_cast<double>(s.m) * static_cast<double>(s.n) * static_cast<double>(s.k_total);
      plan->cls_elems[s.cls] += static_cast<double>(s.m) * static_cast<double>(s.n);
      const uint8_t bit = static_cast<uint8_t>(1u << s.cls);
      // bit 7: read by any MFMA class (the split GEMM runs all of them in one launch)
      constexpr uint8_t kAnyMfma = 0x80;
      const bool mfma = is_mfma_class(s.cls);
      if (mfma) plan->mfma_elems += static_cast<double>(s.m) * static_cast<double>(s.n);
      for (int32_t t = s.t0; t < s.t1; ++t) {
        const ExecTask &e = plan->h_exec[static_cast<size_t>(t)];
        const int64_t ea = int64_t(s.m) * e.k, eb = int64_t(e.k) * s.n;
        uint8_t &wa = seen_a[static_cast<size_t>(e.a_blk)], &wb = seen_b[static_cast<size_t>(e.b_blk)];
        if (wa == 0) plan->a_unique_elems += ea;
        if (wb == 0) plan->b_unique_elems += eb;
        if (!(wa & bit)) plan->cls_elems[s.cls] += static_cast<double>(ea);
        if (!(wb & bit)) plan->cls_elems[s.cls] += static_cast<double>(eb);
        if (mfma && !(wa & kAnyMfma)) plan->mfma_elems += static_cast<double>(ea);
        if (mfma && !(wb & kAnyMfma)) plan->mfma_elems += static_cast<double>(eb);
        wa |= bit | (mfma ? kAnyMfma : 0);
        wb |= bit | (mfma ? kAnyMfma : 0);
      }
    }
  }
  plan->panels_enabled = g_row_panels.load() != 0;
  QLT_TRY(build_tiles(plan.get(), hb));

  // ---- the work list to the device: one allocation, one copy ----
  Packer wl;
  auto bytes_of = [](const auto &v) { return sizeof(v[0]) * v.size(); };
  const size_t w_exec = wl.add(bytes_of(plan->h_exec)), w_segs = wl.add(bytes_of(segs)), w_tiles = wl.add(bytes_of(hb.tiles)),
               w_red = wl.add(bytes_of(hb.red)), w_pt = wl.add(bytes_of(hb.ptiles)), w_po = wl.add(bytes_of(hb.pouts)),
               w_pm = wl.add(bytes_of(hb.pterms));
  const size_t wl_bytes = wl.bytes;
  const size_t w_ga = wl.add(sizeof(BlkGather) * na), w_gb = wl.add(sizeof(BlkGather) * nb);
  hipError_t e = hipMalloc(&plan->d_store, wl.bytes);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc (work list)", __FILE__, __LINE__);
  char *const ds = static_cast<char *>(plan->d_store);
  if (plan->part_doubles > 0) QLT_HIP(hipMalloc(&plan->d_part, sizeof(double) * plan->part_doubles));
  QLT_TRY(back.reserve(wl_bytes));
  auto put = [&](size_t off, const auto &v) {
    if (!v.empty()) std::memcpy(back.at<char>(off), v.data(), sizeof(v[0]) * v.size());
    return v.empty() ? nullptr : ds + off;
  };
  plan->d_exec = reinterpret_cast<ExecTask *>(put(w_exec, plan->h_exec));
  plan->d_segs = reinterpret_cast<Seg *>(put(w_segs, segs));
  plan->d_tiles = reinterpret_cast<Tile *>(put(w_tiles, hb.tiles));
  plan->d_red = reinterpret_cast<ReduceItem *>(put(w_red, hb.red));
  plan->d_ptiles = reinterpret_cast<PanelTile *>(put(w_pt, hb.ptiles));
  plan->d_pouts = reinterpret_cast<PanelOut *>(put(w_po, hb.pouts));
  plan->d_pterms = reinterpret_cast<PanelTerm *>(put(w_pm, hb.pterms));
  plan->d_ga = reinterpret_cast<BlkGather *>(ds + w_ga);
  plan->d_gb = reinterpret_cast<BlkGather *>(ds + w_gb);
  QLT_HIP(hipMemcpyAsync(ds, back.at<char>(0), wl_bytes, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_gather_desc, dim3(blocks_for((na + nb) * 2 * QLT_MAX_RANK)), dim3(256), 0, st, d_ad, na, d_bd, nb, args, plan->d_ga,
                     plan->d_gb);
  QLT_HIP(hipGetLastError());
  QLT_HIP(hipStreamSynchronize(st));
  *plan_out = plan.release();
  return QLT_OK;
}

qlt_status qlt_set_row_panels(int32_t enable) {
  QLT_CHECK_ARG(enable == 0 || enable == 1, "qlt_set_row_panels: enable must be 0 or 1");
  g_row_panels.store(enable);
  return QLT_OK;
}

int32_t qlt_get_row_panels(void) { return g_row_panels.load(); }

qlt_status qlt_plan_destroy(qlt_plan *plan) {
  delete plan;   // the destructor releases the device work list
  return QLT_OK;
}

qlt_status qlt_plan_get_info(const qlt_plan *plan, qlt_plan_info *info) {
  QLT_CHECK_ARG(plan != nullptr && info != nullptr, "qlt_plan_get_info: null argument");
  info->n_tasks = static_cast<int64_t>(plan->tasks.size());
  info->n_c_blks = static_cast<int64_t>(plan->c_blk_idx.size());
  info->c_raw_size = plan->c_raw_size;
  info->c_rank = plan->c_rank;
  info->c_is_scalar = plan->c_is_scalar;
  info->sum_mkn = plan->sum_mkn;
  info->n_tiles = plan->n_tiles;
  info->a_unique_elems = plan->a_unique_elems;
  info->b_unique_elems = plan->b_unique_elems;
  info->n_panel_tiles = plan->n_ptiles;
  return QLT_OK;
}

qlt_status qlt_plan_get_tasks(const qlt_plan *plan, qlt_task *tasks) {
  QLT_CHECK_ARG(plan != nullptr, "qlt_plan_get_tasks: null plan");
  if (plan->tasks.empty()) return QLT_OK;
  QLT_CHECK_ARG(tasks != nullptr, "qlt_plan_get_tasks: null output");
  std::memcpy(tasks, plan->tasks.data(), sizeof(qlt_task) * plan->tasks.size());
  return QLT_OK;
}

qlt_status qlt_plan_get_c_blocks(const qlt_plan *plan, int64_t *blk_idx, int64_t *coords, int64_t *dims,
                                 int64_t *offsets) {
  QLT_CHECK_ARG(plan != nullptr, "qlt_plan_get_c_blocks: null plan");
  const size_t n = plan->c_blk_idx.size();
  if (n == 0) return QLT_OK;
  if (blk_idx) std::memcpy(blk_idx, plan->c_blk_idx.data(), 8 * n);
  if (offsets) std::memcpy(offsets, plan->c_offsets.data(), 8 * n);
  if (coords) std::memcpy(coords, plan->c_coords.data(), 8 * plan->c_coords.size());
  if (dims) std::memcpy(dims, plan->c_dims.data(), 8 * plan->c_dims.size());
  return QLT_OK;
}

qlt_status qlt_plan_set_c_offsets(qlt_plan *plan, const int64_t *c_offsets) {
  QLT_REQUIRE_INIT();
  QLT_CHECK_ARG(plan != nullptr, "qlt_plan_set_c_offsets: null plan");
  const int64_t n = static_cast<int64_t>(plan->h_segs.size());
  if (n == 0) return QLT_OK;
  QLT_CHECK_ARG(c_offsets != nullptr, "qlt_plan_set_c_offsets: null offsets");
  bool same = true;
  for (int64_t o = 0; o < n && same; ++o) same = plan->h_segs[o].c_off == c_offsets[o];
  if (same) return QLT_OK;
  // The kernels of an earlier execute of this plan may still be running on a
  // non-blocking stream and read the segment records (and the split tile
  // records, which carry copies of the output offsets): wait for the whole
  // device before the records change.
  QLT_HIP(hipDeviceSynchronize());
  if (plan->c_is_scalar) {
    plan->h_segs[0].c_off = c_offsets[0];
    for (qlt_task &t : plan->tasks) t.c_data_offset = c_offsets[0];
  } else {
    std::vector<int64_t> by_idx_order(plan->c_blk_idx.size());
    for (int64_t o = 0; o < n; ++o) {
      QLT_CHECK_ARG(c_offsets[o] >= 0, "qlt_plan_set_c_offsets: negative offset");
      plan->h_segs[o].c_off = c_offsets[o];
      plan->c_offsets[o] = c_offsets[o];
    }
    for (qlt_task &t : plan->tasks) {
      auto it = std::lower_bound(plan->c_blk_idx.begin(), plan->c_blk_idx.end(), t.c_blk_idx);
      t.c_data_offset = c_offsets[it - plan->c_blk_idx.begin()];
    }
  }
  QLT_HIP(hipMemcpy(plan->d_segs, plan->h_segs.data(), sizeof(Seg) * n, hipMemcpyHostToDevice));
  // the split metadata holds the old offsets: the next split execute rewrites it
  plan->split_dtype = -1;
  plan->split_mode = -1;
  return QLT_OK;
}

}  // extern "C"
