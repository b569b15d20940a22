// Shared host/device helpers of the KvsAll kernels (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <type_traits>

#include "../../include/kge_hip.h"
#include "kge_host.h"

namespace kge {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

// ---- host-side error plumbing -------------------------------------------------------------
int set_error(int code, const char* fmt, ...);
void clear_error();

#define KGE_REQUIRE(cond, code, ...)                      \
  do {                                                    \
    if (!(cond)) return ::kge::set_error(code, __VA_ARGS__); \
  } while (0)

#define KGE_HIP_CHECK(expr)                                                              \
  do {                                                                                   \
    hipError_t _e = (expr);                                                              \
    if (_e != hipSuccess)                                                                \
      return ::kge::set_error(KGE_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(_e)); \
  } while (0)

#define KGE_LAUNCH_CHECK(name)                                                          \
  do {                                                                                  \
    hipError_t _e = hipGetLastError();                                                  \
    if (_e != hipSuccess)                                                               \
      return ::kge::set_error(KGE_ERR_HIP, "launch of %s failed: %s", name, hipGetErrorString(_e)); \
  } while (0)

// ---- few queries against the whole table (kge_few.hip); the caller has asked host::few_topk_applies / few_scores_applies
int few_topk_launch(const float* Q, const float* bias, const void* E, int dtype, const float* scale, int64_t B, int64_t d,
                    int64_t N, int64_t k, float* out_scores, int64_t* out_idx, int apply_sigmoid, void* workspace,
                    hipStream_t st);
int few_scores_launch(const float* Q, const float* bias, const void* E, int dtype, const float* scale, int64_t B, int64_t d,
                      int64_t N, float* out, int64_t ldo, hipStream_t st);
struct GradArgs;
int few_grad_launch(const float* Q, const float* E, int64_t B, int64_t d, int64_t N, const GradArgs& grad, hipStream_t st);

// ---- MFMA 32x32 accumulator layout --------------------------------------------------------
// acc[i] of lane l holds output (row_of(i, l / 32), l % 32).
__device__ __forceinline__ int row_of(int i, int hf) { return ((i >> 2) << 3) + (hf << 2) + (i & 3); }

// The lanes of one wave see each other's LDS writes from here on (a wave's LDS accesses complete in order, so that only the
// compiler has to be told): for kernels whose waves work on LDS rows of their own.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Order-preserving map float -> uint32 (larger float <=> larger key); NaN is not handled.
__device__ __forceinline__ uint32_t f32_to_ordered(float f) {
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ordered_to_f32(uint32_t k) {
  uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(u);
}

// A threshold that every score equal to x beats in a float comparison (`s > just_below(x)` holds for s == x), as
// close below x as that allows.  One step down in the ordered encoding does it except around zero: the neighbour of
// +0 there is -0, which compares EQUAL to it, and the denormals next to them depend on the comparison honouring
// denormals; so for |x| below the smallest normal the answer is minus the smallest normal.  (-inf stays -inf.)
__device__ __forceinline__ float just_below(float x) {
  if (!(x > __uint_as_float(0xff800000u))) return x;                        // -inf, NaN
  if (__builtin_fabsf(x) < 1.17549435e-38f) return -1.17549435e-38f;
  return ordered_to_f32(f32_to_ordered(x) - 1u);
}

// ---- (head, relation) -> filter row: binary search in the sorted key array -----------------------
__device__ __forceinline__ int64_t filter_row(int64_t first, int64_t second, const int64_t* keys, int64_t n_rows,
                                              int64_t num_relations) {
  const int64_t key = first * num_relations + second;
  int64_t lo = 0, hi = n_rows;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < key) lo = mid + 1; else hi = mid;
  }
  return (lo < n_rows && keys[lo] == key) ? lo : -1;
}

// ---- what a training step needs beside its contractions: the filter rows of its pairs, and the outputs that are added to
// cleared.  Work for some workgroups of a launch that comes early anyway (a launch of its own: 4 us of a toy step's 63).
struct StepPrepare {
  const int64_t* hr;
  int64_t B;  // 0: no filter rows
  const int64_t* keys;
  int64_t n_rows, key_mult;
  int64_t* rows;
  float* clear[8];
  int64_t counts[8];  // 0: no such buffer
};
inline unsigned step_prepare_wgs(const StepPrepare& s) {
  int64_t most = s.B;
  for (int64_t n : s.counts) most = n > most ? n : most;
  const int64_t wgs = (most + 255) / 256;
  return (unsigned)(wgs < 256 ? wgs : 256);
}
__device__ __forceinline__ void step_prepare(const StepPrepare& s, unsigned wg, unsigned wgs) {
  const int64_t i0 = (int64_t)wg * blockDim.x + threadIdx.x, stride = (int64_t)wgs * blockDim.x;
  for (int64_t b = i0; b < s.B; b += stride) s.rows[b] = filter_row(s.hr[2 * b], s.hr[2 * b + 1], s.keys, s.n_rows, s.key_mult);
  for (int j = 0; j < 8; ++j)
    for (int64_t i = i0; i < s.counts[j]; i += stride) s.clear[j][i] = 0.f;
}

}  // namespace kge
