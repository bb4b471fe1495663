// Pivot candidates of the LU kernels: keys as unsigned integers in the order
// of the pivot rule (IAMAX with the NaN rule of kernel/arm/iamax.c:51-74), the
// best lane of a wavefront, candidates that carry their position.
#pragma once
#include <hip/hip_runtime.h>

namespace oba {

// pivot key as an unsigned integer whose order is the pivot rule's
template <typename T> struct LuKey;
template <> struct LuKey<float> {
  typedef unsigned U;
  __device__ static inline U key(float x, bool at_j) {
    const unsigned b = __float_as_uint(x) & 0x7fffffffu;
    return b > 0x7f800000u ? (at_j ? 0x7f800001u : 0u) : b + 1u;
  }
};
template <> struct LuKey<double> {
  typedef unsigned long long U;
  __device__ static inline U key(double x, bool at_j) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x) & 0x7fffffffffffffffull;
    return b > 0x7ff0000000000000ull ? (at_j ? 0x7ff0000000000001ull : 0ull) : b + 1ull;
  }
};

template <int CTRL>
__device__ __attribute__((always_inline)) inline unsigned l3_dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
// wavefront maximum of an unsigned, uniform
__device__ __attribute__((always_inline)) inline unsigned l3_wave_max(unsigned v) {
  v = max(v, l3_dpp<0xB1>(v));
  v = max(v, l3_dpp<0x4E>(v));
  v = max(v, l3_dpp<0x141>(v));
  v = max(v, l3_dpp<0x140>(v));
  const unsigned a = max((unsigned)__builtin_amdgcn_readlane((int)v, 0), (unsigned)__builtin_amdgcn_readlane((int)v, 16));
  const unsigned b = max((unsigned)__builtin_amdgcn_readlane((int)v, 32), (unsigned)__builtin_amdgcn_readlane((int)v, 48));
  return max(a, b);
}
// The lane holding the best candidate, uniform: the largest key, ties to the
// lowest position; npos is the complemented position (larger is lower).  The
// lanes that share the largest word are almost always one.
__device__ __attribute__((always_inline)) inline int l3_tie(unsigned long long m, unsigned npos) {
  const bool in = (m >> (threadIdx.x & 63)) & 1;   // the lanes of m compete by position
  const unsigned c = in ? npos : 0u;
  const unsigned mx = l3_wave_max(c);
  return __builtin_ctzll(__ballot(in && c == mx));
}
__device__ __attribute__((always_inline)) inline int l3_best_lane(unsigned key, unsigned npos) {
  const unsigned mx = l3_wave_max(key);
  const unsigned long long m = __ballot(key == mx);
  if (__popcll(m) == 1) return __builtin_ctzll(m);
  return l3_tie(m, npos);
}
__device__ __attribute__((always_inline)) inline int l3_best_lane(unsigned long long key, unsigned npos) {
  const unsigned hi = (unsigned)(key >> 32);
  const unsigned mx = l3_wave_max(hi);
  unsigned long long m = __ballot(hi == mx);
  if (__popcll(m) == 1) return __builtin_ctzll(m);
  const unsigned lo = hi == mx ? (unsigned)key : 0u;
  const unsigned ml = l3_wave_max(lo);
  m = __ballot(hi == mx && lo == ml);
  if (__popcll(m) == 1) return __builtin_ctzll(m);
  return l3_tie(m, npos);
}
__device__ __attribute__((always_inline)) inline unsigned l3_rl(unsigned v, int l) { return (unsigned)__builtin_amdgcn_readlane((int)v, l); }
__device__ __attribute__((always_inline)) inline unsigned long long l3_rl(unsigned long long v, int l) {
  return ((unsigned long long)l3_rl((unsigned)(v >> 32), l) << 32) | l3_rl((unsigned)v, l);
}
__device__ __attribute__((always_inline)) inline float l3_rlf(float v, int l) { return __uint_as_float(l3_rl(__float_as_uint(v), l)); }
__device__ __attribute__((always_inline)) inline double l3_rlf(double v, int l) { return __longlong_as_double((long long)l3_rl((unsigned long long)__double_as_longlong(v), l)); }

// one candidate in an order that an unsigned comparison decides: larger key,
// then lower position (kept complemented)
template <typename T> struct LuCand;
template <> struct LuCand<float> {
  unsigned npos, key;
  __device__ inline unsigned long long v() const { return ((unsigned long long)key << 32) | npos; }
  __device__ inline bool beats(const LuCand& o) const { return v() > o.v(); }
};
template <> struct __attribute__((aligned(16))) LuCand<double> {
  unsigned long long key;
  unsigned npos, pad;
  __device__ inline bool beats(const LuCand& o) const { return (key > o.key) | ((key == o.key) & (npos > o.npos)); }
};

}  // namespace oba
