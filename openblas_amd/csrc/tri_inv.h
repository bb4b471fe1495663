// Inverse of a 64x64 lower triangle in LDS: 16x16 blocks by substitution, joins
// on the matrix cores.  A matrix element (i, k) is at k*(TRI_NB + 1) + i.  What a
// wavefront leaves in LDS other lanes of it may read after a wave_fence().
#pragma once
#include <hip/hip_runtime.h>
#include "wave.h"

namespace oba {

constexpr int TRI_NB = 64;

// lane K of each row of 16 lanes, to all of the row
template <int K>
__device__ inline float tri_bcast16(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xF, 0xF, false));
}
template <int K>
__device__ inline double tri_bcast16(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + K, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + K, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
template <int K, typename T>
__device__ __attribute__((always_inline)) inline void tri_inv16_step(T (&y)[4], const T (&l)[16], T r, int i, int g) {
  if constexpr (K < 15) {
    const T rk = tri_bcast16<K>(r);
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const T f = y[c] - l[K] * (tri_bcast16<K>(y[c]) * rk);
      y[c] = i > K && K >= g + 4 * c ? f : y[c];   // an Inf or NaN of L only meets terms that there are
    }
    tri_inv16_step<K + 1>(y, l, r, i, g);
  }
}
// One wavefront inverts the 16x16 lower triangle at o (diagonal reciprocals
// in rinv): lane (i, g) = (lane % 16, lane / 16) holds row i of columns g,
// g+4, g+8, g+12; row k, once final, reaches the rows below by DPP row
// broadcasts.
template <typename T>
__device__ __attribute__((always_inline)) inline void tri_inv16(const T* S, T* Y, const T* rinv, int o) {
  constexpr int LD = TRI_NB + 1;
  const int i = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
  T l[16], y[4];
#pragma unroll
  for (int k = 0; k < 16; k++) l[k] = S[(o + k) * LD + o + i];
  const T r = rinv[o + i];
#pragma unroll
  for (int c = 0; c < 4; c++) y[c] = i == g + 4 * c ? T(1) : T(0);
  tri_inv16_step<0>(y, l, r, i, g);
#pragma unroll
  for (int c = 0; c < 4; c++) Y[(o + g + 4 * c) * LD + o + i] = i >= g + 4 * c ? y[c] * r : T(0);
}

// one wavefront: tile (ri, ci) of `o` = sign * sum over the 16-deep tiles k0
// .. k0+NK of x(ri, k) y(k, ci), in 64x64 LDS matrices
template <int NK, typename T>
__device__ __attribute__((always_inline)) inline void tri_prod(T* o, const T* x, const T* y, int ri, int ci, int k0,
                                                                 T sign) {
  constexpr int LD = TRI_NB + 1;
  typedef MF<T> mf;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  typename mf::acc acc[2] = {};
#pragma unroll
  for (int k = 0; k < 16 * NK; k += 4)
    acc[(k >> 2) & 1] = mf::mma(y[(16 * ci + lr) * LD + 16 * k0 + k + lg], x[(16 * k0 + k + lg) * LD + 16 * ri + lr],
                                acc[(k >> 2) & 1]);
  acc[0] += acc[1];
#pragma unroll
  for (int r = 0; r < 4; r++) o[(16 * ci + mf::orow(lane, r)) * LD + 16 * ri + lr] = sign * acc[0][r];
}

}  // namespace oba
