// Helpers of a single wavefront.
#pragma once
#include <hip/hip_runtime.h>

namespace oba {

// Between LDS stores of some lanes and loads of them by others of the same
// wavefront: the hardware keeps a wavefront's LDS accesses in order, this keeps
// the compiler from moving one over the other.  No instruction.
__device__ __attribute__((always_inline)) inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

}  // namespace oba
