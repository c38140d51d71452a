// Scalar helpers and shared pieces of the batched dense decompositions
// (block_svd.hip, block_qr.hip): real and complex elements behind one set of
// overloads.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "qlt_internal.h"

namespace qlt {
namespace dense {

typedef double v4d __attribute__((ext_vector_type(4)));

struct cplx {
  double x, y;
};

__device__ __forceinline__ double re_(double a) { return a; }
__device__ __forceinline__ double re_(cplx a) { return a.x; }
__device__ __forceinline__ double conj_(double a) { return a; }
__device__ __forceinline__ cplx conj_(cplx a) { return {a.x, -a.y}; }
__device__ __forceinline__ double mul_(double a, double b) { return a * b; }
__device__ __forceinline__ cplx mul_(cplx a, cplx b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// conj(a) * b
__device__ __forceinline__ double cmul_(double a, double b) { return a * b; }
__device__ __forceinline__ cplx cmul_(cplx a, cplx b) { return {a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x}; }
__device__ __forceinline__ double add_(double a, double b) { return a + b; }
__device__ __forceinline__ cplx add_(cplx a, cplx b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ double sub_(double a, double b) { return a - b; }
__device__ __forceinline__ cplx sub_(cplx a, cplx b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ double scl_(double s, double a) { return s * a; }
__device__ __forceinline__ cplx scl_(double s, cplx a) { return {s * a.x, s * a.y}; }
__device__ __forceinline__ double abs2_(double a) { return a * a; }
__device__ __forceinline__ double abs2_(cplx a) { return a.x * a.x + a.y * a.y; }
template <typename T> __device__ __forceinline__ T zero_();
template <> __device__ __forceinline__ double zero_<double>() { return 0.0; }
template <> __device__ __forceinline__ cplx zero_<cplx>() { return {0.0, 0.0}; }
template <typename T> __device__ __forceinline__ T one_();
template <> __device__ __forceinline__ double one_<double>() { return 1.0; }
template <> __device__ __forceinline__ cplx one_<cplx>() { return {1.0, 0.0}; }
// unit phase of g (|g| > 0), conjugated: e^{-i arg g}, from 1 / |g|
__device__ __forceinline__ double uphase_conj_inv(double g, double inv) { return g * inv; }
__device__ __forceinline__ cplx uphase_conj_inv(cplx g, double inv) { return {g.x * inv, -g.y * inv}; }
// complex reciprocal
__device__ __forceinline__ double recip_(double a) { return 1.0 / a; }
__device__ __forceinline__ cplx recip_(cplx a) {
  const double d = a.x * a.x + a.y * a.y;
  return {a.x / d, -a.y / d};
}

template <bool C> struct ElemOf { using T = double; };
template <> struct ElemOf<true> { using T = cplx; };

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ double shfl_(double v, int src) { return __shfl(v, src); }
__device__ __forceinline__ cplx shfl_(cplx v, int src) { return {__shfl(v.x, src), __shfl(v.y, src)}; }
__device__ __forceinline__ double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// Device allocation released at scope exit.
struct DevBuf {
  void *p = nullptr;
  ~DevBuf() {
    if (p != nullptr) (void)hipFree(p);
  }
};

inline qlt_status check_shapes(const char *who, int64_t n_mats, const int64_t *rows, const int64_t *cols) {
  QLT_CHECK_ARG(n_mats >= 0, std::string(who) + ": negative matrix count");
  QLT_CHECK_ARG(n_mats == 0 || (rows != nullptr && cols != nullptr), std::string(who) + ": null shape array");
  QLT_CHECK_ARG(n_mats < (int64_t(1) << 31), std::string(who) + ": too many matrices");
  for (int64_t i = 0; i < n_mats; ++i)
    QLT_CHECK_ARG(rows[i] >= 1 && cols[i] >= 1, std::string(who) + ": matrix " + std::to_string(i) + " is empty");
  return QLT_OK;
}

// Extent (elements) of a buffer addressed by offsets.  Single-precision
// element types are widened to FP64 (complex128) device buffers, decomposed
// there, and the factors rounded back.
inline int64_t extent(int64_t n, const int64_t *offs, const int64_t *r, const int64_t *c) {
  int64_t e = 0;
  for (int64_t i = 0; i < n; ++i) e = offs[i] + r[i] * c[i] > e ? offs[i] + r[i] * c[i] : e;
  return e;
}

}  // namespace dense
}  // namespace qlt
