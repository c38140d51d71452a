// Device-resident Krylov primitives over a basis arena: block inner products,
// block updates and the Lanczos extension step, with the number of active
// basis vectors kept in device memory.  They let one Lanczos iteration --
// the matvec chain, two passes of classical Gram-Schmidt against the whole
// basis, the normalisation of the new vector -- be launched with no host
// round trip, so it can be captured once as a graph and replayed.  They
// restate the vector operations the reference's Lanczos solver uses on
// tensors: InnerProduct (tensor_manipulation/basic_operations.h:146-203),
// LinearCombine (ten_linear_combine.h:186) and Normalize
// (qltensor/qltensor_impl.h:568-573), on raw data.
//
// Every reduction is two-pass with a fixed grid and a fixed summation order,
// so results are bitwise reproducible (a replayed graph equals the eager
// launches bit for bit).

#include <algorithm>
#include <cmath>
#include <string>

#include "qlt_internal.h"

namespace {

constexpr int kParts = 512;          // partial sums per reduction (fixed grid)
constexpr int kSweep = 16;           // basis vectors a sweep over w reads together
constexpr int32_t kMaxBasis = 1024;  // arena slots a call may address

__device__ __forceinline__ int active_count(const int32_t *count, int32_t k_max) {
  const int m = *count;
  return m < 0 ? 0 : (m > k_max ? k_max : m);
}

// Sum over the 256 threads of a workgroup, in a fixed order: wave shuffles,
// then the four wave sums in order.  Every thread gets the result.
__device__ __forceinline__ double block_sum(double v, double *s_red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int tid = threadIdx.x;
  __syncthreads();
  if ((tid & 63) == 0) s_red[tid >> 6] = v;
  __syncthreads();
  return ((s_red[0] + s_red[1]) + s_red[2]) + s_red[3];
}

template <bool CPLX>
__device__ __forceinline__ double2 elem(const double *__restrict__ x, int64_t e) {
  if (CPLX) return reinterpret_cast<const double2 *>(x)[e];
  return double2{x[e], 0.0};
}

template <bool CPLX>
__device__ __forceinline__ void put_elem(double *__restrict__ x, int64_t e, double2 y) {
  if (CPLX) reinterpret_cast<double2 *>(x)[e] = y;
  else x[e] = y.x;
}

// One sweep of a workgroup over its elements of w (grid stride: the same
// elements and the same threads in every kernel of kParts workgroups).
//
// UPDATE: w[e] += sum_{i < m} c_i V_i[e], the terms added in order of i
// (s_c: the scaled coefficients).  DOT: the workgroup's partial products
// work[(i * kParts + b) * 2 + {0, 1}] = sum conj(V_i) w of the vectors
// i0 <= i < min(i0 + NQ, m); with UPDATE of the updated w, m <= NQ and
// i0 = 0, from the basis values already read.  NORM: returns the thread's
// sum of |w[e]|^2.  The fused multiply-adds are written out: left to the
// compiler, two instances may round a complex term differently.
//
// What bounds it: the reads of V at the sizes of a large bond; below some
// 10^6 elements the latency of one element's loads, which go out NQ at a
// time (a vector past the count reads the first one and is not used), and
// the tree of sums at the end.  Its NQ wave reductions run interleaved, with
// one barrier for all of them: with two barriers per product (the sums one
// after the other) the sums of 16 products were half of the kernel.  Update
// and 16 products of 2 * 10^5 FP64 elements, with the final sums: 15.7 ->
// 12.3 us; of 8 * 10^6: 223 -> 218 us (5 TB/s).  The loads of several
// elements at a time gave nothing more (12.2, 217).
template <bool CPLX, int NQ, bool UPDATE, bool DOT, bool NORM>
__device__ __forceinline__ double sweep(int64_t n, int i0, int m, const double *s_c, const double *__restrict__ V,
                                        int64_t ldv, double *__restrict__ w, double *work, double (*s_red)[4]) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t first = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  double ar[NQ], ai[NQ], norm = 0.0;
#pragma unroll
  for (int q = 0; q < NQ; ++q) ar[q] = ai[q] = 0.0;
  for (int64_t e = first; e < n; e += stride) {
    double2 y = elem<CPLX>(w, e);
    double2 x[NQ];
    for (int g = i0; g < m; g += NQ) {
      const int nq = min(NQ, m - g);
#pragma unroll
      for (int q = 0; q < NQ; ++q) x[q] = elem<CPLX>(V + (g + (q < nq ? q : 0)) * ldv * (CPLX ? 2 : 1), e);
      if (!UPDATE) break;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        if (q < nq) {
          const double cr = s_c[2 * (g + q)], ci = s_c[2 * (g + q) + 1];
          if (CPLX) {
            y.x = fma(-ci, x[q].y, fma(cr, x[q].x, y.x));
            y.y = fma(ci, x[q].x, fma(cr, x[q].y, y.y));
          } else {
            y.x = fma(cr, x[q].x, y.x);
          }
        }
      }
    }
    if (UPDATE) put_elem<CPLX>(w, e, y);
    if (DOT) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        if (q < m - i0) {
          if (CPLX) {
            ar[q] = fma(x[q].y, y.y, fma(x[q].x, y.x, ar[q]));
            ai[q] = fma(-x[q].y, y.x, fma(x[q].x, y.y, ai[q]));
          } else {
            ar[q] = fma(x[q].x, y.x, ar[q]);
          }
        }
      }
    }
    if (NORM) norm = CPLX ? fma(y.y, y.y, fma(y.x, y.x, norm)) : fma(y.x, y.x, norm);
  }
  if (DOT) {
    // each product's sum in the order of block_sum
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        ar[q] += __shfl_down(ar[q], off, 64);
        if (CPLX) ai[q] += __shfl_down(ai[q], off, 64);
      }
    }
    const int tid = threadIdx.x;
    __syncthreads();
    if ((tid & 63) == 0) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        s_red[2 * q][tid >> 6] = ar[q];
        s_red[2 * q + 1][tid >> 6] = ai[q];
      }
    }
    __syncthreads();
    if (tid < 2 * min(NQ, m - i0)) {
      const double *r = s_red[tid];
      work[(static_cast<int64_t>(i0 + (tid >> 1)) * kParts + blockIdx.x) * 2 + (tid & 1)] =
          ((r[0] + r[1]) + r[2]) + r[3];
    }
  }
  return norm;
}

// The narrowest sweep over the vectors left: loads and sums of vectors past
// the count are not free (2 products of 10^6 complex elements in a sweep of 8:
// 15.7 us, of 2: 12.2).
// An update in FP64 by up to half as many vectors again as kSweep takes them in
// halves for the same reason: by 17 vectors of 3 * 10^6 elements 92.9 -> 87.8 us,
// by 20 of 2 * 10^5 7.5 -> 6.6 (complex, and more vectors: no difference).
template <bool CPLX, bool UPDATE, bool DOT, bool NORM>
__device__ __forceinline__ double sweep_of(int64_t n, int i0, int m, const double *s_c, const double *__restrict__ V,
                                           int64_t ldv, double *__restrict__ w, double *work, double (*s_red)[4]) {
  if (UPDATE && !DOT && !CPLX && m > kSweep && m <= kSweep + kSweep / 2)
    return sweep<CPLX, kSweep / 2, UPDATE, DOT, NORM>(n, i0, m, s_c, V, ldv, w, work, s_red);
  if (m - i0 <= kSweep / 8)
    return sweep<CPLX, kSweep / 8, UPDATE, DOT, NORM>(n, i0, m, s_c, V, ldv, w, work, s_red);
  if (m - i0 <= kSweep / 4)
    return sweep<CPLX, kSweep / 4, UPDATE, DOT, NORM>(n, i0, m, s_c, V, ldv, w, work, s_red);
  if (m - i0 <= kSweep / 2)
    return sweep<CPLX, kSweep / 2, UPDATE, DOT, NORM>(n, i0, m, s_c, V, ldv, w, work, s_red);
  return sweep<CPLX, kSweep, UPDATE, DOT, NORM>(n, i0, m, s_c, V, ldv, w, work, s_red);
}

template <bool CPLX>
__device__ __forceinline__ void dot_sweeps(int64_t n, int m, const double *__restrict__ V, int64_t ldv,
                                           double *__restrict__ w, double *work, double (*s_red)[4]) {
  for (int i0 = 0; i0 < m; i0 += kSweep)
    sweep_of<CPLX, false, true, false>(n, i0, m, nullptr, V, ldv, w, work, s_red);
}

__device__ __forceinline__ void scaled_coefs(double *s_c, int m, double scale, const double *__restrict__ c) {
  for (int i = threadIdx.x; i < m; i += blockDim.x) {
    s_c[2 * i] = scale * c[2 * i];
    s_c[2 * i + 1] = scale * c[2 * i + 1];
  }
  __syncthreads();
}

// work[(i * kParts + b) * 2 + {0, 1}] = partial <V_i, w> of workgroup b
// (conj(V_i) * w), for i < m.
template <bool CPLX>
__global__ __launch_bounds__(256) void k_basis_dot_partial(int64_t n, int32_t k_max, const int32_t *count,
                                                           const double *__restrict__ V, int64_t ldv, double *w,
                                                           double *work) {
  __shared__ double s_red[2 * kSweep][4];
  dot_sweeps<CPLX>(n, active_count(count, k_max), V, ldv, w, work, s_red);
}

// c[2i], c[2i+1] = sum over the partials of basis vector i (i < m), else 0.
// One workgroup per basis vector.
__global__ __launch_bounds__(256) void k_basis_dot_final(int32_t k_max, const int32_t *count,
                                                         const double *work, double *c) {
  __shared__ double s_red[4];
  const int i = blockIdx.x;
  const int m = active_count(count, k_max);
  double sr = 0.0, si = 0.0;
  if (i < m) {
    for (int b = threadIdx.x; b < kParts; b += blockDim.x) {
      sr += work[(static_cast<int64_t>(i) * kParts + b) * 2];
      si += work[(static_cast<int64_t>(i) * kParts + b) * 2 + 1];
    }
  }
  sr = block_sum(sr, s_red);
  si = block_sum(si, s_red);
  if (threadIdx.x == 0) {
    c[2 * i] = sr;
    c[2 * i + 1] = si;
  }
}

// w[e] += scale * sum_{i < m} c_i V_i[e], the terms added in order of i.
template <bool CPLX>
__global__ __launch_bounds__(256) void k_basis_update(int64_t n, int32_t k_max, const int32_t *count, double scale,
                                                      const double *__restrict__ c, const double *__restrict__ V,
                                                      int64_t ldv, double *__restrict__ w) {
  __shared__ double s_c[2 * kMaxBasis];
  const int m = active_count(count, k_max);
  scaled_coefs(s_c, m, scale, c);
  sweep_of<CPLX, true, false, false>(n, 0, m, s_c, V, ldv, w, nullptr, nullptr);
}

// The update of k_basis_update followed by the partial products of
// k_basis_dot_partial on the updated w, in one pass over the basis when
// m <= kSweep: each thread keeps its elements' basis values between the two.
// With more vectors the products follow in sweeps of their own, each thread
// reading back the elements of w that it wrote.  The same terms in the same
// order per element and per partial sum, so w and the partials are bitwise
// those of the two kernels run one after the other.
template <bool CPLX>
__global__ __launch_bounds__(256) void k_basis_update_dot(int64_t n, int32_t k_max, const int32_t *count,
                                                          double scale, const double *__restrict__ c,
                                                          const double *__restrict__ V, int64_t ldv,
                                                          double *__restrict__ w, double *work) {
  __shared__ double s_c[2 * kMaxBasis];
  __shared__ double s_red[2 * kSweep][4];
  const int m = active_count(count, k_max);
  scaled_coefs(s_c, m, scale, c);
  if (m <= kSweep) {
    sweep_of<CPLX, true, true, false>(n, 0, m, s_c, V, ldv, w, work, s_red);
  } else {
    sweep_of<CPLX, true, false, false>(n, 0, m, s_c, V, ldv, w, nullptr, nullptr);
    dot_sweeps<CPLX>(n, m, V, ldv, w, work, s_red);
  }
}

// work[b] = partial sum of |w_e|^2 of workgroup b, of w updated as by
// k_basis_update when UPDATE (a pass over w and a launch less than the two
// kernels); work[kParts] = m, from which k_lanczos_store takes the count
// that it advances.
template <bool CPLX, bool UPDATE>
__global__ __launch_bounds__(256) void k_norm2_partial(int64_t n, int32_t k_max, const int32_t *count, double scale,
                                                       const double *__restrict__ c, const double *__restrict__ V,
                                                       int64_t ldv, double *__restrict__ w, double *work) {
  __shared__ double s_c[UPDATE ? 2 * kMaxBasis : 1];
  __shared__ double s_red[4];
  const int m = active_count(count, k_max);
  double acc;
  if (UPDATE) {
    scaled_coefs(s_c, m, scale, c);
    acc = sweep_of<CPLX, true, false, true>(n, 0, m, s_c, V, ldv, w, nullptr, nullptr);
  } else {
    acc = sweep<CPLX, 1, false, false, true>(n, 0, 0, nullptr, V, ldv, w, nullptr, nullptr);
  }
  acc = block_sum(acc, s_red);
  if (threadIdx.x == 0) {
    work[blockIdx.x] = acc;
    if (blockIdx.x == 0) work[kParts] = m;
  }
}

// The Lanczos coefficients of vector j = m - 1, alpha_j = Re c_j and beta_j =
// |w|; V_m = w / beta_j (0 when beta_j = 0) and m = m + 1 when slot m exists
// (m < k_max).  Every workgroup sums the kParts partials of |w|^2 itself, in
// one order; m is the one k_norm2_partial saw, so that workgroup 0 may
// advance the count.  (As launches of their own the coefficients and the
// count took 3.6 and 2.5 us of an iteration; 16 iterations at U(1) D = 1024 in FP64,
// with the update's norm: 2.77 -> 2.60 ms.)
template <bool CPLX>
__global__ __launch_bounds__(256) void k_lanczos_store(int64_t n, int32_t k_max, int32_t *count,
                                                       const double *__restrict__ c, const double *__restrict__ work,
                                                       const double *__restrict__ w, double *__restrict__ V,
                                                       int64_t ldv, double *alphas, double *betas) {
  __shared__ double s_red[4];
  const int m = static_cast<int>(work[kParts]);
  double acc = 0.0;
  for (int b = threadIdx.x; b < kParts; b += blockDim.x) acc += work[b];
  const double beta = sqrt(block_sum(acc, s_red));
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (m > 0) {
      alphas[m - 1] = c[2 * (m - 1)];
      betas[m - 1] = beta;
    }
    if (m < k_max) *count = m + 1;
  }
  if (m >= k_max) return;
  const double inv = beta > 0.0 ? 1.0 / beta : 0.0;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; e < n; e += stride) {
    const double2 y = elem<CPLX>(w, e);
    put_elem<CPLX>(V + m * ldv * (CPLX ? 2 : 1), e, double2{y.x * inv, y.y * inv});
  }
}

// x = V_{*index + offset} (nothing when that slot is outside 0 .. k_max - 1).
template <bool CPLX>
__global__ __launch_bounds__(256) void k_basis_select(int64_t n, int32_t k_max, const int32_t *index, int32_t offset,
                                                      const double *__restrict__ V, int64_t ldv,
                                                      double *__restrict__ x) {
  const int s = *index + offset;
  if (s < 0 || s >= k_max) return;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; e < n; e += stride) {
    if (CPLX) reinterpret_cast<double2 *>(x)[e] = reinterpret_cast<const double2 *>(V)[s * ldv + e];
    else x[e] = V[s * ldv + e];
  }
}

inline unsigned stream_grid(int64_t n) {
  return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 8192)));
}

qlt_status check_basis_args(const char *fn, int32_t dtype, int64_t n, int32_t k_max, int64_t ldv) {
  using qlt::fail;
  QLT_CHECK_ARG(dtype == QLT_F64 || dtype == QLT_C128, std::string(fn) + ": bad dtype");
  QLT_CHECK_ARG(n >= 0, std::string(fn) + ": negative length");
  QLT_CHECK_ARG(k_max >= 1 && k_max <= kMaxBasis, std::string(fn) + ": k_max must be in 1 .. 1024");
  QLT_CHECK_ARG(ldv >= n, std::string(fn) + ": slot stride below the vector length");
  return QLT_OK;
}

// |w| (of w updated by scale * c_update first, when c_update is given), the
// coefficients, V_m and the count.
void launch_extend(int32_t dtype, int64_t n, int32_t k_max, int32_t *count, const double *c, double scale,
                   const double *c_update, double *w, double *V, int64_t ldv, double *alphas, double *betas,
                   double *work, hipStream_t st) {
  const bool cplx = dtype == QLT_C128;
  const auto norm = c_update ? (cplx ? k_norm2_partial<true, true> : k_norm2_partial<false, true>)
                             : (cplx ? k_norm2_partial<true, false> : k_norm2_partial<false, false>);
  hipLaunchKernelGGL(norm, dim3(kParts), dim3(256), 0, st, n, k_max, count, scale, c_update, V, ldv, w, work);
  const unsigned grid = std::min(stream_grid(n), 2u * kParts);   // each workgroup sums the partials
  hipLaunchKernelGGL(cplx ? k_lanczos_store<true> : k_lanczos_store<false>, dim3(grid), dim3(256), 0, st, n, k_max,
                     count, c, work, w, V, ldv, alphas, betas);
}

}  // namespace

using namespace qlt;

extern "C" {

qlt_status qlt_basis_dot(int32_t dtype, int64_t n, int32_t k_max, const int32_t *count, const void *V, int64_t ldv,
                         const void *w, double *c, double *work, void *stream) {
  QLT_REQUIRE_INIT();
  QLT_TRY(check_basis_args("qlt_basis_dot", dtype, n, k_max, ldv));
  QLT_CHECK_ARG(count && V && w && c && work, "qlt_basis_dot: null pointer");
  hipStream_t st = as_stream(stream);
  const auto *vd = static_cast<const double *>(V);
  auto *wd = const_cast<double *>(static_cast<const double *>(w));   // only read
  hipLaunchKernelGGL(dtype == QLT_C128 ? k_basis_dot_partial<true> : k_basis_dot_partial<false>, dim3(kParts),
                     dim3(256), 0, st, n, k_max, count, vd, ldv, wd, work);
  hipLaunchKernelGGL(k_basis_dot_final, dim3(k_max), dim3(256), 0, st, k_max, count, work, c);
  QLT_HIP(hipGetLastError());
  return QLT_OK;
}

qlt_status qlt_basis_update_dot(int32_t dtype, int64_t n, int32_t k_max, const int32_t *count, double scale,
                                const double *c, const void *V, int64_t ldv, void *w, double *c_out, double *work,
                                void *stream) {
  QLT_REQUIRE_INIT();
  QLT_TRY(check_basis_args("qlt_basis_update_dot", dtype, n, k_max, ldv));
  QLT_CHECK_ARG(count && V && w && c && c_out && work, "qlt_basis_update_dot: null pointer");
  QLT_CHECK_ARG(c != c_out, "qlt_basis_update_dot: c and c_out must not alias");
  hipStream_t st = as_stream(stream);
  const auto *vd = static_cast<const double *>(V);
  auto *wd = static_cast<double *>(w);
  hipLaunchKernelGGL(dtype == QLT_C128 ? k_basis_update_dot<true> : k_basis_update_dot<false>, dim3(kParts),
                     dim3(256), 0, st, n, k_max, count, scale, c, vd, ldv, wd, work);
  hipLaunchKernelGGL(k_basis_dot_final, dim3(k_max), dim3(256), 0, st, k_max, count, work, c_out);
  QLT_HIP(hipGetLastError());
  return QLT_OK;
}

qlt_status qlt_basis_update(int32_t dtype, int64_t n, int32_t k_max, const int32_t *count, double scale,
                            const double *c, const void *V, int64_t ldv, void *w, void *stream) {
  QLT_REQUIRE_INIT();
  QLT_TRY(check_basis_args("qlt_basis_update", dtype, n, k_max, ldv));
  QLT_CHECK_ARG(count && V && w && c, "qlt_basis_update: null pointer");
  if (n == 0) return QLT_OK;
  hipStream_t st = as_stream(stream);
  const auto *vd = static_cast<const double *>(V);
  auto *wd = static_cast<double *>(w);
  if (dtype == QLT_C128)
    hipLaunchKernelGGL(k_basis_update<true>, dim3(stream_grid(n)), dim3(256), 0, st, n, k_max, count, scale, c, vd,
                       ldv, wd);
  else
    hipLaunchKernelGGL(k_basis_update<false>, dim3(stream_grid(n)), dim3(256), 0, st, n, k_max, count, scale, c, vd,
                       ldv, wd);
  QLT_HIP(hipGetLastError());
  return QLT_OK;
}

qlt_status qlt_lanczos_extend(int32_t dtype, int64_t n, int32_t k_max, int32_t *count, const double *c,
                              const void *w, void *V, int64_t ldv, double *alphas, double *betas, double *work,
                              void *stream) {
  QLT_REQUIRE_INIT();
  QLT_TRY(check_basis_args("qlt_lanczos_extend", dtype, n, k_max, ldv));
  QLT_CHECK_ARG(count && c && w && V && alphas && betas && work, "qlt_lanczos_extend: null pointer");
  auto *wd = const_cast<double *>(static_cast<const double *>(w));   // only read without an update
  launch_extend(dtype, n, k_max, count, c, 0.0, nullptr, wd, static_cast<double *>(V), ldv, alphas, betas, work,
                as_stream(stream));
  QLT_HIP(hipGetLastError());
  return QLT_OK;
}

qlt_status qlt_lanczos_update_extend(int32_t dtype, int64_t n, int32_t k_max, int32_t *count, const double *c,
                                     double scale, const double *c_update, void *w, void *V, int64_t ldv,
                                     double *alphas, double *betas, double *work, void *stream) {
  QLT_REQUIRE_INIT();
  QLT_TRY(check_basis_args("qlt_lanczos_update_extend", dtype, n, k_max, ldv));
  QLT_CHECK_ARG(count && c && c_update && w && V && alphas && betas && work,
                "qlt_lanczos_update_extend: null pointer");
  launch_extend(dtype, n, k_max, count, c, scale, c_update, static_cast<double *>(w), static_cast<double *>(V), ldv,
                alphas, betas, work, as_stream(stream));
  QLT_HIP(hipGetLastError());
  return QLT_OK;
}

qlt_status qlt_basis_select(int32_t dtype, int64_t n, int32_t k_max, const int32_t *index, int32_t offset,
                            const void *V, int64_t ldv, void *x, void *stream) {
  QLT_REQUIRE_INIT();
  QLT_TRY(check_basis_args("qlt_basis_select", dtype, n, k_max, ldv));
  QLT_CHECK_ARG(index && V && x, "qlt_basis_select: null pointer");
  if (n == 0) return QLT_OK;
  hipStream_t st = as_stream(stream);
  const auto *vd = static_cast<const double *>(V);
  auto *xd = static_cast<double *>(x);
  if (dtype == QLT_C128)
    hipLaunchKernelGGL(k_basis_select<true>, dim3(stream_grid(n)), dim3(256), 0, st, n, k_max, index, offset, vd, ldv,
                       xd);
  else
    hipLaunchKernelGGL(k_basis_select<false>, dim3(stream_grid(n)), dim3(256), 0, st, n, k_max, index, offset, vd,
                       ldv, xd);
  QLT_HIP(hipGetLastError());
  return QLT_OK;
}

}  // extern "C"
