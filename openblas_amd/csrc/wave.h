// Helpers of a single wavefront, shared by the kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace oba {

// The 16x16x4 matrix instructions: lane l gives row l%16, k = l/16 of the first
// operand and column l%16, k = l/16 of the second; accumulator element r of
// lane l is row orow(l, r), column l%16 (measured; FP64 and FP32 differ).
template <typename T> struct MF;
template <> struct MF<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  __device__ static inline acc mma(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ static inline int orow(int l, int r) { return 4 * r + (l >> 4); }
};
template <> struct MF<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  __device__ static inline acc mma(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  __device__ static inline int orow(int l, int r) { return 4 * (l >> 4) + r; }
};

// Between LDS stores of some lanes and loads of them by others of the same
// wavefront: the hardware keeps a wavefront's LDS accesses in order, this keeps
// the compiler from moving one over the other.  No instruction.
__device__ __attribute__((always_inline)) inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

}  // namespace oba
