// Device code shared by the ray kernels (ray_program.hip, ray_column.hip):
// the sign function of the reference's JAX semantics and detector binning.
#pragma once

#include "tg_common.hpp"

namespace tgr {

template <typename T>
__device__ __forceinline__ T sign_of(T a) {
  if (a != a || a == T(0)) return a;
  return a > T(0) ? T(1) : T(-1);
}

// Pixel index of one position; -1 when it falls outside the detector.
__device__ __forceinline__ int64_t bin_index(const tg_bin_spec& B, double y, double x) {
  // Same operation order as apply_transformation's T @ [y, x, 1]
  // (reference coordinate_transforms.py:104-140), in f64.
  const double fy = __dadd_rn(__dadd_rn(__dmul_rn(B.m[0], y), __dmul_rn(B.m[1], x)), B.m[2]);
  const double fx = __dadd_rn(__dadd_rn(__dmul_rn(B.m[3], y), __dmul_rn(B.m[4], x)), B.m[5]);
  // jnp.round is round-half-to-even; rint uses the default RNE mode.
  const int32_t iy = tg::xla_f64_to_i32(rint(fy));
  const int32_t ix = tg::xla_f64_to_i32(rint(fx));
  if (iy < 0 || iy >= B.height || ix < 0 || ix >= B.width) return -1;
  return (int64_t)iy * B.width + ix;
}

template <typename T>
__device__ __forceinline__ void global_deposit(const tg_bin_spec& B, int64_t p, T w) {
  switch (B.acc_dtype) {
    case 0:
      atomicAdd((int32_t*)B.acc + p, 1);
      break;
    case 1:
      atomicAdd((unsigned long long*)B.acc + p, 1ull);
      break;
    case 2:
      unsafeAtomicAdd((float*)B.acc + p, (float)w);
      break;
    default:
      unsafeAtomicAdd((double*)B.acc + p, (double)w);
      break;
  }
}

// A workgroup's private histogram: packed 16-bit counters in LDS, two bins per
// 32-bit word.  A workgroup may count at most kMaxRaysPerGroup rays, so a
// counter never carries into its neighbour.
constexpr int64_t kMaxRaysPerGroup = 65535;
// Largest private histogram: the CU's 160 KB of LDS.  A 256x256 detector
// (128 KB) counts here too; with memory atomics 1M rays on 3,600 of its bins
// took 179 us, as atomics on one cache line execute one after another.
constexpr int64_t kLdsBins = 81920;

// LDS words of a histogram of nb bins (whole 16-byte groups, which lds_clear
// writes at once).
__host__ __device__ __forceinline__ int64_t lds_words(int64_t nb) { return (nb + 7) / 8 * 4; }

// Dynamic LDS beyond 64 KB has to be asked for.
inline int allow_lds(const void* kernel, size_t bytes) {
  if (bytes > 65536)
    TG_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return TG_OK;
}

template <int NT>
__device__ __forceinline__ void lds_clear(int32_t* hist, int nb) {
  for (int i = threadIdx.x; i < (nb + 7) / 8; i += NT) ((int4*)hist)[i] = make_int4(0, 0, 0, 0);
}

__device__ __forceinline__ void lds_deposit(int32_t* hist, int64_t p) {
  atomicAdd(&hist[p >> 1], 1 << (16 * (int)(p & 1)));
}

// Adds a private histogram of the bins [first_bin, first_bin + nb) into the
// accumulator.  The cost is the cache lines each atomic instruction touches,
// hardly the lanes in it, so the lanes of a wavefront take consecutive bins
// (a lane unpacking both bins of its word touched every line twice).  Each
// workgroup starts at a place of its own: all of them starting at bin 0 meet
// on the same lines (a flush of 256 workgroups over 57,600 bins took 88 us in
// step, 46 us so).
template <int NT>
__device__ __forceinline__ void lds_flush(const tg_bin_spec& B, const int32_t* hist, int64_t first_bin, int nb) {
  // a wavefront takes 512 bins at a time, 16 bytes a lane, to skip what is empty
  const int lane = threadIdx.x & 63, groups = (nb + 511) / 512, quads = (nb + 7) / 8;
  const int turn = (int)((int64_t)groups * blockIdx.x / gridDim.x);
  for (int k = threadIdx.x >> 6; k < groups; k += NT / 64) {
    const int g = k + turn < groups ? k + turn : k + turn - groups;
    const int4 q = g * 64 + lane < quads ? ((const int4*)hist)[g * 64 + lane] : make_int4(0, 0, 0, 0);
    const uint64_t used = __ballot((q.x | q.y | q.z | q.w) != 0);
    for (int j = 0; j < 8; ++j) {
      if (((used >> (8 * j)) & 0xff) == 0) continue;
      const int i = g * 512 + j * 64 + lane;
      if (i >= nb) continue;
      const int32_t c = (int32_t)(((uint32_t)hist[i >> 1] >> (16 * (i & 1))) & 0xffffu);
      if (c == 0) continue;
      if (B.acc_dtype == 0)
        atomicAdd((int32_t*)B.acc + first_bin + i, c);
      else
        atomicAdd((unsigned long long*)B.acc + first_bin + i, (unsigned long long)(int64_t)c);
    }
  }
}

}  // namespace tgr
