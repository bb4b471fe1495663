// One BM x BN tile of C = alpha*op(A)*op(B) + beta*C by 4 wavefronts: operand
// slabs, the main loop and the store, shared by the GEMM and the batched GEMM
// kernels (design notes in gemm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include "wave.h"

namespace oba {

// A vector of V elements at an element-aligned (not 16-byte-aligned) address:
// global loads and stores of 16 bytes only need 4-byte alignment, so odd
// leading dimensions and tiles that start anywhere use the same wide accesses
// (with per-element loads 2047 x 3001 x 1501 FP64 took 606 us).
template <typename T, int V> struct UVec { typedef T type __attribute__((ext_vector_type(V), aligned(sizeof(T)))); };
template <typename T, int V> struct AVec { typedef T type __attribute__((ext_vector_type(V))); };

// Loads one BK-deep slab of an operand tile (TILE along m or n) into
// registers.  KC: the operand is contiguous along k in memory (Trans A /
// NoTrans B).  The slab is staged k-major in LDS, s[BK][TILE + 4]: a lane
// reads V consecutive m (n) of one k with one 16-byte read, and the padding
// spreads the k-strided writes of a KC operand over the banks.
template <typename T, int TILE, int BK, bool KC>
struct TileLoader {
  static constexpr int V = 16 / sizeof(T);
  static constexpr int NV = TILE * BK / V / 256;  // vectors per thread
  static_assert(NV * V * 256 == TILE * BK, "tile must divide over 256 threads");
  static constexpr int LD = TILE + 4;
  static constexpr int SIZE = BK * LD;   // elements per buffer
  typedef typename AVec<T, V>::type vec;
  vec r[NV];

  // FULL: the whole slab is in range.  Otherwise (an operand narrower than the
  // tile or the slab) rows past MN repeat the last one (their results are
  // never stored) and k past K gives zeros; the addresses are clamped, so no
  // load is predicated.
  template <bool FULL>
  __device__ inline void load(const T* __restrict__ g, long ld, long mn0, long k0, long MN, long K) {
    const int tid = threadIdx.x & 255;   // thread within its 256-thread group
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int v = tid + i * 256;
      long mn, k;
      if (!KC) { k = v / (TILE / V); mn = (v % (TILE / V)) * V; }
      else { mn = v / (BK / V); k = (v % (BK / V)) * V; }
      mn += mn0; k += k0;
      if constexpr (FULL) {
        r[i] = *(const typename UVec<T, V>::type*)(KC ? g + k + mn * ld : g + mn + k * ld);
      } else {
#pragma unroll
        for (int e = 0; e < V; e++) {
          const long mm = min(KC ? mn : mn + e, MN - 1), kk = KC ? k + e : k, kc = min(kk, K - 1);
          const T x = g[KC ? kc + mm * ld : mm + kc * ld];
          r[i][e] = kk < K ? x : T(0);
        }
      }
    }
  }
  // The K tail is read as the last BK of the operand's k, where every load is
  // in range; this clears the first kmin of it, which the slab before had (in
  // both operands: an infinity must not meet the other's zero).
  __device__ inline void clear(int kmin) {
    const int tid = threadIdx.x & 255;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int v = tid + i * 256, k = KC ? (v % (BK / V)) * V : v / (TILE / V);
#pragma unroll
      for (int e = 0; e < V; e++) r[i][e] = (KC ? k + e : k) < kmin ? T(0) : r[i][e];
    }
  }
  __device__ inline void zero() {
#pragma unroll
    for (int i = 0; i < NV; i++) r[i] = vec{};
  }
  // writes the slab into its LDS buffer (layout above)
  __device__ inline void store(T* s) const {
    const int tid = threadIdx.x & 255;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int v = tid + i * 256;
      if (!KC) {
        const int k = v / (TILE / V), mn = (v % (TILE / V)) * V;
        *(vec*)(s + k * LD + mn) = r[i];
      } else {
        const int mn = v / (BK / V), k = (v % (BK / V)) * V;
#pragma unroll
        for (int e = 0; e < V; e++) s[(k + e) * LD + mn] = r[i][e];
      }
    }
  }
};

template <typename T, int BM, int BN, int BK, bool TA, bool TB>
struct GemmTile {
  typedef TileLoader<T, BM, BK, TA> LA;
  typedef TileLoader<T, BN, BK, !TB> LB;
  static constexpr int V = LA::V, BK_ = BK;
  static constexpr int WTM = BM / 2, WTN = BN / 2;  // 2x2 waves
  static constexpr int FM = WTM / 16, FN = WTN / 16;
  // fragment i of a wave's tile holds rows PM*(lane%16) + i%PM of the
  // i/PM-th group of 16*PM rows, so one LDS read feeds PM fragments and a
  // lane's outputs are PM consecutive rows of C (likewise PN columns of B)
  static constexpr int PM = FM < V ? FM : V, PN = FN < V ? FN : V;
  // a wave with a single fragment runs its k steps through 4 accumulators in
  // turn: independent MFMAs instead of one dependent chain, and shorter sums
  static constexpr int NA = FM * FN == 1 ? 4 : 1;
  typedef MF<T> mf;
  typedef typename mf::acc acc_t;
  // a tail moved back into range costs registers around the loop: not for 128-
  // wide tiles, whose K is long (FP32 8192^3 0.5 % slower with it)
  static constexpr bool MOVE_TAIL = BM * BN <= 64 * 64;
  static constexpr int STAGE = 2 * (LA::SIZE + LB::SIZE);   // double-buffered slabs, elements of LDS

  // acc = the tile's product over nk slabs, rows from m0 and columns from n0
  // (in range where the operand is as wide as the tile); st: STAGE elements
  static __device__ __attribute__((always_inline)) inline void product(acc_t (&acc)[FM][FN], long M, long N, long K,
                                                                       const T* __restrict__ A, long lda,
                                                                       const T* __restrict__ B, long ldb, long m0,
                                                                       long n0, int nk, T* st) {
    // buffer b of the A slab at st + b*LA::SIZE, of the B slab after both A's
#define OBA_AS(b) (st + (b) * LA::SIZE)
#define OBA_BS(b) (st + 2 * LA::SIZE + (b) * LB::SIZE)
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
    const int wm0 = (wave & 1) * WTM, wn0 = (wave >> 1) * WTN;
    LA la;
    LB lb;

    acc_t accs[NA][FM][FN];
#pragma unroll
    for (int q = 0; q < NA; q++)
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) accs[q][i][j] = acc_t{};
    // A slab's fragments are read from LDS into registers one slab ahead, so
    // the reads run behind the MFMAs of the slab before instead of in front of
    // their own.
    struct Frags {
      T a[BK / 4][FM], b[BK / 4][FN];
    };
    Frags f0, f1;
    auto read = [&](int buf, Frags& f) __attribute__((always_inline)) {
      const T* as = OBA_AS(buf) + wm0;
      const T* bs = OBA_BS(buf) + wn0;
#pragma unroll
      for (int kk = 0; kk < BK / 4; kk++) {
        const int kr = kk * 4 + (lane >> 4);
#pragma unroll
        for (int i = 0; i < FM; i += PM)
          *(typename AVec<T, PM>::type*)&f.a[kk][i] =
              *(const typename AVec<T, PM>::type*)&as[kr * LA::LD + i * 16 + PM * (lane & 15)];
#pragma unroll
        for (int j = 0; j < FN; j += PN)
          *(typename AVec<T, PN>::type*)&f.b[kk][j] =
              *(const typename AVec<T, PN>::type*)&bs[kr * LB::LD + j * 16 + PN * (lane & 15)];
      }
    };
    auto mma = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
      for (int kk = 0; kk < BK / 4; kk++)
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
          for (int j = 0; j < FN; j++)
            accs[kk % NA][i][j] = mf::mma(f.b[kk][j], f.a[kk][i], accs[kk % NA][i][j]);
    };
    // A slab that lies in range is loaded unconditionally, an operand narrower
    // than the tile (or a K below one slab) through clamped addresses; the K
    // tail moves back into range.  With sliced K a group past its range's end multiplies zeros,
    // so that all groups meet the same barriers.
    const bool fit_a = M >= BM, fit_b = N >= BN, fits = fit_a && fit_b;
    auto fetch = [&](long k0) __attribute__((always_inline)) {
      if (k0 >= K) {
        la.zero();
        lb.zero();
        return;
      }
      const bool in = k0 + BK <= K, tail = MOVE_TAIL && !in && K >= BK;
      const long kb = tail ? K - BK : k0;
      if (fit_a && (in || tail)) la.template load<true>(A, lda, m0, kb, M, K);
      else la.template load<false>(A, lda, m0, kb, M, K);
      if (fit_b && (in || tail)) lb.template load<true>(B, ldb, n0, kb, N, K);
      else lb.template load<false>(B, ldb, n0, kb, N, K);
      if (tail) {
        la.clear((int)(k0 - kb));
        lb.clear((int)(k0 - kb));
      }
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
      la.store(OBA_AS(buf));
      lb.store(OBA_BS(buf));
    };
    const int nfull = fits ? (int)(K / BK) : 0;   // leading slabs that lie in range
    fetch(0);
    stage(0);
    fetch(BK);
    __syncthreads();
    read(0, f0);
    int kt = 0;
    // one step: slab kt+1 from registers to LDS, slab kt+2 from memory to
    // registers, slab kt+1's fragments read while slab kt is multiplied.  No
    // control flow around the loads of a slab in range, so that they stay in
    // flight across the MFMAs.
    auto step = [&](auto full_tag, int buf, Frags& cur, Frags& next) __attribute__((always_inline)) {
      stage(buf);
      if constexpr (decltype(full_tag)::value) {
        la.template load<true>(A, lda, m0, (long)(kt + 2) * BK, M, K);
        lb.template load<true>(B, ldb, n0, (long)(kt + 2) * BK, N, K);
      } else {
        fetch((long)(kt + 2) * BK);
      }
      __syncthreads();
      read(buf, next);
      mma(cur);
      kt++;
    };
    while (kt + 3 < nfull) {
      step(std::true_type{}, 1, f0, f1);
      step(std::true_type{}, 0, f1, f0);
    }
    while (kt + 2 < nk) {
      step(std::false_type{}, 1, f0, f1);
      step(std::false_type{}, 0, f1, f0);
    }
    if (kt + 1 < nk) {   // kt is even: slab kt in f0, slab kt+1 in registers
      stage(1);
      __syncthreads();
      read(1, f1);
      mma(f0);
      mma(f1);
    } else if (kt < nk) {
      mma(f0);
    }
    if constexpr (NA == 4) accs[0][0][0] = (accs[0][0][0] + accs[1][0][0]) + (accs[2][0][0] + accs[3][0][0]);
#undef OBA_AS
#undef OBA_BS
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++) acc[i][j] = accs[0][i][j];
  }

  // the tile owns C rows from mt and columns from nt, computed from m0, n0 on;
  // tri 1 (2): only the lower (upper) triangle of C is written
  static __device__ __attribute__((always_inline)) inline void store(const acc_t (&acc)[FM][FN], long M, long N, T alpha,
                                                                     T beta, T* __restrict__ C, long ldc, long mt,
                                                                     long nt, long m0, long n0, int tri) {
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
    const int wm0 = (wave & 1) * WTM, wn0 = (wave >> 1) * WTN;
    const bool bz = (beta == T(0)), fits = M >= BM && N >= BN;
    // a tile whose every element is its own to write: PM rows per store
    const bool whole = m0 == mt && n0 == nt && fits && (tri == 0 || (tri == 1 ? m0 >= n0 + BN - 1 : m0 + BM - 1 <= n0));
    typedef typename UVec<T, PM>::type uvec;
    if (whole) {
#pragma unroll
      for (int i = 0; i < FM; i += PM) {
        T* const pc = C + m0 + wm0 + i * 16 + PM * (lane & 15) + (n0 + wn0) * ldc;
#pragma unroll
        for (int j = 0; j < FN; j++) {
          uvec old[4];
          T* p[4];
#pragma unroll
          for (int r = 0; r < 4; r++) {
            p[r] = pc + ((j / PN) * 16 * PN + PN * mf::orow(lane, r) + j % PN) * ldc;
            if (!bz) old[r] = *(const uvec*)p[r];
          }
#pragma unroll
          for (int r = 0; r < 4; r++) {
            uvec v;
#pragma unroll
            for (int e = 0; e < PM; e++) {
              v[e] = alpha * acc[i + e][j][r];
              if (!bz) v[e] += beta * old[r][e];
            }
            *(uvec*)p[r] = v;
          }
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < FM; i++) {
      const long m = m0 + wm0 + (i / PM) * 16 * PM + PM * (lane & 15) + i % PM;
#pragma unroll
      for (int j = 0; j < FN; j++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const long n = n0 + wn0 + (j / PN) * 16 * PN + PN * mf::orow(lane, r) + j % PN;
          if (m >= mt && n >= nt && m < M && n < N && !(tri == 1 && n > m) && !(tri == 2 && m > n)) {
            T* p = C + m + n * ldc;
            T v = alpha * acc[i][j][r];
            if (!bz) v += beta * *p;
            *p = v;
          }
        }
      }
    }
  }
};

}  // namespace oba
