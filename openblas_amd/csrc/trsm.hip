// Triangular solve with multiple right-hand sides (all 8 side/uplo/trans
// forms, unit or non-unit diagonal), device pointers, column-major.
//
// Reference semantics: B <- alpha*B first (driver/level3/trsm_L.c:103-107;
// alpha == 0 zeroes B and returns), then op(A)*X = B (left) or X*op(A) = B
// (right), the diagonal applied as a multiplication by its reciprocal
// (kernel/generic/trsm_ltcopy_2.c:43 INV(a) = 1/a, trsm_kernel_LT.c:95).
//
// Design: recursive blocking on the triangle (split in halves on a 64-row
// grid) so that almost all flops land in large MFMA GEMM updates.  Leaves (up
// to 256 rows or columns of the triangle) are substitutions on the left side
// and multiply by explicit inverses of the 64x64 diagonal blocks on the right.
// A left-side triangle of a single block is solved by wavefronts of
// right-hand-side vectors: lane i owns x_i and row i of the triangle, and x_k is
// broadcast with v_readlane after it is final (forward or backward
// column-oriented substitution).
#include "kernels.h"
#include "tri_inv.h"

namespace oba {

constexpr int TRSM_NB = 64;

__device__ inline double bcast_lane(double v, int k) {
  int lo = __builtin_amdgcn_readlane(__double2loint(v), k);
  int hi = __builtin_amdgcn_readlane(__double2hiint(v), k);
  return __hiloint2double(hi, lo);
}
__device__ inline float bcast_lane(float v, int k) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}

// Solves E x = b for nvec vectors, E = op(A), nb <= 64.  Element i of vector v
// lies at B[i + v*ldb].  eT: E(i,k) = A(k,i) (else A(i,k)); elower: E is lower
// triangular.  A wavefront per vector (two, interleaved, halve the workgroups:
// DTRSM 8192 x 1024 3.52 ms against 3.21 when its leaves were these).
template <typename T>
__global__ __launch_bounds__(256) void trsm_leaf_kernel(int nb, long nvec, const T* __restrict__ A, long lda,
                                                        T* __restrict__ B, long ldb, bool eT, bool elower, bool unit,
                                                        const int* abort_flag) {
  constexpr int LDE = TRSM_NB + 1;     // padded: conflict-free transposed stores
  __shared__ T E[TRSM_NB * LDE];       // E(i,k) at E[k*LDE + i]
  __shared__ T dinv[TRSM_NB];
  if (abort_flag && *abort_flag) return;
  // consecutive threads read consecutive addresses of A in both layouts;
  // every load issued before the first LDS write (clamped in-bounds
  // addresses, the padding selected after)
  constexpr int SU = TRSM_NB * TRSM_NB / 256;
  T sv[SU];
#pragma unroll
  for (int u = 0; u < SU; u++) {
    const int idx = threadIdx.x + 256 * u, f = idx & 63, s = idx >> 6;   // f: fast (contiguous) index of A
    sv[u] = A[min(f, nb - 1) + (long)min(s, nb - 1) * lda];
  }
#pragma unroll
  for (int u = 0; u < SU; u++) {
    const int idx = threadIdx.x + 256 * u, f = idx & 63, s = idx >> 6;
    // eT: E(i,k) = A(k,i) -> A[f + s*lda] = A(f, s) = E(s, f)
    const int i = eT ? s : f, k = eT ? f : s;
    E[k * LDE + i] = (f < nb && s < nb) ? sv[u] : T(0);
  }
  __syncthreads();
  if (threadIdx.x < TRSM_NB) {
    const int k = threadIdx.x;
    dinv[k] = (k < nb && !unit) ? T(1) / E[k * LDE + k] : T(1);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const long v = (long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  // lane i holds row i of E and its reciprocal pivot in registers; the steps
  // are unrolled (static register indices; a runtime step loop reading E from
  // LDS inside the chain took ~36 us per 64 x 1024 leaf)
  T e[TRSM_NB];
#pragma unroll
  for (int k = 0; k < TRSM_NB; k++) e[k] = E[k * LDE + lane];
  const T di = dinv[lane];
  T x = (v < nvec && lane < nb) ? B[v * ldb + lane] : T(0);
  if (elower) {
#pragma unroll
    for (int k = 0; k < TRSM_NB; k++) {
      if (k < nb) {
        if (lane == k) x *= di;
        const T xk = bcast_lane(x, k);
        if (lane > k) x -= e[k] * xk;
      }
    }
  } else {
#pragma unroll
    for (int k = TRSM_NB - 1; k >= 0; k--) {
      if (k < nb) {
        if (lane == k) x *= di;
        const T xk = bcast_lane(x, k);
        if (lane < k) x -= e[k] * xk;
      }
    }
  }
  if (v < nvec && lane < nb) B[v * ldb + lane] = x;
}

// Leaves of up to TRSM_RN rows or columns of the triangle in one launch: the
// right side through explicit inverses of the 64x64 diagonal blocks, the left
// side by substitution.  (A fully unrolled per-row substitution on the right
// side is ~4000 straight-line instructions run once per wavefront and measured
// at 40-65 us per leaf whatever its size, instruction fetch.)
//
// (1) One workgroup per diagonal block b of M = op(A) (upper or lower,
//     unit or not) computes M_bb^{-1} by doubling, as the lower triangle L =
//     M or M^T: the four 16x16 diagonal blocks by substitution, one per
//     wavefront (tri_inv.h; the diagonal applied as a multiplication by its
//     reciprocal as trsm_kernel_LT.c:95), then pairs joined with two products
//     each on the matrix cores, Y21 = -Y22 (L21 Y11), 16 -> 32 -> 64.  Stored
//     row-major at inv[b*64*64 + i*64 + j].  The bound is the chain of 16
//     substitution steps and four products: 7.8 us FP64 with its launch; 12.9 with a thread per
//     column reading L from LDS and the joins on the vector unit.
template <typename T>
__global__ __launch_bounds__(256) void trsm_inv_diag_kernel(long na, const T* __restrict__ A, long lda, bool mT,
                                                            bool mupper, bool unit, T* __restrict__ inv,
                                                            const int* abort_flag) {
  constexpr int LD = TRI_NB + 1;
  __shared__ T S[TRSM_NB * LD];   // L, the other triangle zero
  __shared__ T Y[TRSM_NB * LD];   // its inverse
  __shared__ T U[TRSM_NB * LD];   // products of the joins
  __shared__ T s_rinv[TRSM_NB];
  if (abort_flag && *abort_flag) return;
  const long o = (long)blockIdx.x * TRSM_NB;
  const int nb = (int)min((long)TRSM_NB, na - o);
  const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool flip = mT != mupper;   // L(i,k) = A(k,i)
  // staging: every load issued before the first LDS write (unconditional
  // loads from clamped, in-bounds addresses; the padding is selected after)
  constexpr int SU = TRSM_NB * TRSM_NB / 256;
  T sv[SU];
#pragma unroll
  for (int u = 0; u < SU; u++) {
    const int idx = t + 256 * u, f = idx & 63, g = idx >> 6;   // A(o+f, o+g), f contiguous
    sv[u] = A[(o + min(f, nb - 1)) + (o + min(g, nb - 1)) * lda];
  }
#pragma unroll
  for (int u = 0; u < SU; u++) {
    const int idx = t + 256 * u, f = idx & 63, g = idx >> 6;
    const int i = flip ? g : f, k = flip ? f : g;
    const bool in = i < nb && k < nb;
    S[k * LD + i] = i > k && in ? sv[u] : T(0);
    Y[k * LD + i] = T(0);
    if (i == k) s_rinv[i] = in && !unit ? T(1) / sv[u] : T(1);   // padded with the identity
  }
  __syncthreads();
  tri_inv16(S, Y, s_rinv, 16 * w);
  __syncthreads();
  if (w < 2) {
    tri_prod<1>(U, S, Y, 2 * w + 1, 2 * w, 2 * w, T(1));
    wave_fence();
    tri_prod<1>(Y, Y, U, 2 * w + 1, 2 * w, 2 * w + 1, T(-1));
  }
  __syncthreads();
  tri_prod<2>(U, S, Y, 2 + (w >> 1), w & 1, 0, T(1));
  __syncthreads();
  tri_prod<2>(Y, Y, U, 2 + (w >> 1), w & 1, 2, T(-1));
  __syncthreads();
  T* out = inv + (long)blockIdx.x * TRSM_NB * TRSM_NB;
  for (int idx = t; idx < TRSM_NB * TRSM_NB; idx += 256) {
    const int i = idx >> 6, j = idx & 63;
    out[idx] = (i < nb && j < nb) ? (mupper ? Y[i * LD + j] : Y[j * LD + i]) : T(0);
  }
}

// (2) One launch solves X M = B for up to TRSM_RN columns, in place: a
//     workgroup owns RB rows of B in LDS and takes the 64-column blocks in
//     dependency order, X_b = (B_b - sum_k X_k M_kb) M_bb^{-1}, the products
//     on the matrix cores (wavefront w: columns 16w..16w+15 of the block).
//     The tiles of M and of the inverses come straight from L2 as fragments,
//     the next tile's loads in flight behind the current one's MFMAs; step s
//     of a product takes k = 16*(lane/16) + s, so a lane's 16 elements of M
//     are consecutive in memory where M's columns are.  Rows never meet, so
//     there is no exchange between workgroups; the bound is the chain of tile
//     products (10 of them and 8 barriers at 256 columns).  A call with the
//     inversion and ~10 us of launch, against the recursion of 64-column
//     multiplies and GEMMs (2 N/64 - 1 launches) that this replaced: 64 x 256
//     FP64 90.0 -> 41.6 us, FP32 73.5 -> 35.2; 16000 x 256 116 -> 72, 83 -> 50;
//     4000 x 2000 1056 -> 461, 739 -> 322.
constexpr int TRSM_RN = 256;

template <typename T, int RB, bool MT>
__global__ __launch_bounds__(256) void trsm_right_kernel(int n, long nvec, const T* __restrict__ A, long lda,
                                                         bool upper, const T* __restrict__ inv, T* __restrict__ B,
                                                         long ldb, const int* abort_flag) {
  constexpr int LDX = RB + 2, RT = RB / 16, NB = TRSM_NB;
  typedef MF<T> mf;
  __shared__ T Xs[TRSM_RN * LDX];   // X(r, c) at Xs[c*LDX + r]
  __shared__ T Ts[NB * LDX];        // B_b less the products of the solved blocks
  if (abort_flag && *abort_flag) return;
  const long v0 = (long)blockIdx.x * RB;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), lr = lane & 15, lg = lane >> 4;
  const int nblk = (n + NB - 1) / NB, np = nblk * NB;
  const int rows = (int)min((long)RB, nvec - v0);
  auto blk_of = [&](int q) { return upper ? q : nblk - 1 - q; };
  // tile (q, p): p < q: M(block p, block q) of the order of solution; p == q: the inverse of block q
  auto fetch = [&](int q, int p, T (&f)[16]) __attribute__((always_inline)) {
    const int b = blk_of(q), c = 16 * w + lr;
    if (p == q) {
      const T* src = inv + (long)b * NB * NB + 16 * lg * NB + c;
#pragma unroll
      for (int s = 0; s < 16; s++) f[s] = src[s * NB];
      return;
    }
    const int k0 = blk_of(p) * NB + 16 * lg, cc = b * NB + c;
    if ((b + 1 < nblk && blk_of(p) + 1 < nblk) || np == n) {   // whole tiles
#pragma unroll
      for (int s = 0; s < 16; s++) f[s] = MT ? A[cc + (long)(k0 + s) * lda] : A[k0 + s + (long)cc * lda];
    } else {
#pragma unroll
      for (int s = 0; s < 16; s++) {
        const int k = min(k0 + s, n - 1), ce = min(cc, n - 1);
        const T x = MT ? A[ce + (long)k * lda] : A[k + (long)ce * lda];
        f[s] = k0 + s < n && cc < n ? x : T(0);
      }
    }
  };
  T cur[16], next[16];
  fetch(0, 0, next);
  for (int i0 = 0; i0 < np * RB; i0 += 256 * 16) {
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int i = i0 + t + 256 * u, r = i % RB, c = i / RB;
      v[u] = B[v0 + min(r, rows - 1) + (long)min(c, n - 1) * ldb];
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int i = i0 + t + 256 * u, r = i % RB, c = i / RB;
      if (c < np) Xs[c * LDX + r] = c < n && r < rows ? v[u] : T(0);
    }
  }
  __syncthreads();
  typename mf::acc acc[RT];
#pragma unroll
  for (int i = 0; i < RT; i++) acc[i] = typename mf::acc{};
  int q = 0, p = 0;
  while (true) {
#pragma unroll
    for (int s = 0; s < 16; s++) cur[s] = next[s];
    int nq = q, np2 = p + 1;
    if (np2 > q) { nq = q + 1; np2 = 0; }
    if (nq < nblk) fetch(nq, np2, next);
    const int b = blk_of(q);
    T* const xb = Xs + b * NB * LDX;
    if (p == q) {   // T = B_b - products, every wavefront its 16 columns
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int x = 0; x < 4; x++) {
          const int o = (16 * w + mf::orow(lane, x)) * LDX + 16 * i + lr;
          Ts[o] = xb[o] - acc[i][x];
          acc[i][x] = T(0);
        }
      __syncthreads();
    }
    const T* src = (p == q ? Ts : Xs + blk_of(p) * NB * LDX) + 16 * lg * LDX + lr;
#pragma unroll
    for (int s = 0; s < 16; s++)
#pragma unroll
      for (int i = 0; i < RT; i++) acc[i] = mf::mma(cur[s], src[s * LDX + 16 * i], acc[i]);
    if (p == q) {   // X_b to LDS and memory
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int x = 0; x < 4; x++) {
          const int c = 16 * w + mf::orow(lane, x), r = 16 * i + lr;
          xb[c * LDX + r] = acc[i][x];
          if (r < rows && b * NB + c < n) B[v0 + r + (long)(b * NB + c) * ldb] = acc[i][x];
          acc[i][x] = T(0);
        }
      if (nq >= nblk) break;
      __syncthreads();
    }
    q = nq;
    p = np2;
  }
}

// x[0..N-1] += (y of lane K of each 16-lane row) * e[0..N-1], the broadcast
// taken by the FMA itself; the leading s_nop covers the wait states between a
// VALU write of y and its DPP read
#define TRSM_DPP(T, D, Y, E, K) "v_fmac_" T "_dpp %" #D ", %" #Y ", %" #E " row_newbcast:%" #K " row_mask:0xf bank_mask:0xf\n\t"
#define TRSM_AXPY(TY, T)                                                                                              \
  template <int K, int N>                                                                                             \
  __device__ __attribute__((always_inline)) inline void trsm_axpy(TY* x, TY y, const TY* e) {                         \
    if constexpr (N == 4)                                                                                             \
      asm("s_nop 1\n\t" TRSM_DPP(T, 0, 4, 5, 9) TRSM_DPP(T, 1, 4, 6, 9) TRSM_DPP(T, 2, 4, 7, 9) TRSM_DPP(T, 3, 4, 8, 9) \
          : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]), "+&v"(x[3])                                                        \
          : "v"(y), "v"(e[0]), "v"(e[1]), "v"(e[2]), "v"(e[3]), "n"(K));                                              \
    else if constexpr (N == 3)                                                                                        \
      asm("s_nop 1\n\t" TRSM_DPP(T, 0, 3, 4, 7) TRSM_DPP(T, 1, 3, 5, 7) TRSM_DPP(T, 2, 3, 6, 7)                       \
          : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]) : "v"(y), "v"(e[0]), "v"(e[1]), "v"(e[2]), "n"(K));                  \
    else if constexpr (N == 2)                                                                                        \
      asm("s_nop 1\n\t" TRSM_DPP(T, 0, 2, 3, 5) TRSM_DPP(T, 1, 2, 4, 5)                                               \
          : "+&v"(x[0]), "+&v"(x[1]) : "v"(y), "v"(e[0]), "v"(e[1]), "n"(K));                                          \
    else if constexpr (N == 1)                                                                                        \
      asm("s_nop 1\n\t" TRSM_DPP(T, 0, 1, 2, 3) : "+&v"(x[0]) : "v"(y), "v"(e[0]), "n"(K));                           \
  }
TRSM_AXPY(double, "f64")
TRSM_AXPY(float, "f32")
#undef TRSM_AXPY
#undef TRSM_DPP

// rows i, 16+i, ... of columns TRSM_SG*G.. of a 64x64 lower triangle E (E + i given)
constexpr int TRSM_SG = 4;
template <int G, typename T>
__device__ __attribute__((always_inline)) inline void trsm_subst_read(T (&ec)[TRSM_SG][4], const T* e) {
#pragma unroll
  for (int c = 0; c < TRSM_SG; c++)
#pragma unroll
    for (int s = TRSM_SG * G / 16; s < 4; s++) ec[c][s] = e[(TRSM_SG * G + c) * (TRSM_NB + 1) + 16 * s];
}
// column C and the later ones of its group; x[v][s]: rows 16s+i less the
// columns so far, nr[s] the negative reciprocals of their diagonal
template <int C, int NV, typename T>
__device__ __attribute__((always_inline)) inline void trsm_subst_col(T (&x)[NV][4], T (&sol)[NV][4], const T (&nr)[4],
                                                                     const T (&ec)[TRSM_SG][4], int i) {
  constexpr int S = C / 16, K = C % 16, S1 = K == 15 ? S + 1 : S;   // the last row of a step has none below it there
#pragma unroll
  for (int v = 0; v < NV; v++) {
    // solved rows of the step take the column too: their solution is kept
    // apart, and nothing reads x of a solved row
    const T y = x[v][S] * nr[S];
    sol[v][S] = i == K ? y : sol[v][S];
    trsm_axpy<K, 4 - S1>(x[v] + S1, y, ec[C % TRSM_SG] + S1);
  }
  if constexpr ((C + 1) % TRSM_SG != 0) trsm_subst_col<C + 1>(x, sol, nr, ec, i);
}
template <int G, int NV, typename T>
__device__ __attribute__((always_inline)) inline void trsm_subst_group(T (&x)[NV][4], T (&sol)[NV][4], const T (&nr)[4],
                                                                       const T (&ec)[TRSM_SG][4], const T* e, int i) {
  if constexpr (G + 1 < TRSM_NB / TRSM_SG) {
    T en[TRSM_SG][4];
    trsm_subst_read<G + 1>(en, e);
    __builtin_amdgcn_sched_barrier(0);   // the next group's reads run behind this one's chain
    trsm_subst_col<TRSM_SG * G>(x, sol, nr, ec, i);
    __builtin_amdgcn_sched_barrier(0);
    trsm_subst_group<G + 1>(x, sol, nr, en, e, i);
  } else {
    trsm_subst_col<TRSM_SG * G>(x, sol, nr, ec, i);
  }
}
// One wavefront solves the 64x64 lower triangle E (E(i, k) at E[k*65 + i], its
// diagonal's reciprocals apart in rinv) for 4 NV vectors in place: lane (i, g)
// = (lane % 16, lane / 16) holds rows i, 16+i, 32+i and 48+i of vectors g, g+4,
// ...  A row, once final, reaches the later ones by DPP inside the FMAs, so no
// row leaves its wavefront and there is no barrier inside; an Inf or NaN stays
// with the rows that depend on it.  The element (k, v) lies at xm[k*si + v] and
// the reciprocal k at rinv[k*ri] (both strides negative: the rows of an upper
// triangle, counted from its end).  The bound is the chain of 64 columns, a
// multiplication and an FMA each.
template <int NV, typename T>
__device__ __attribute__((always_inline)) inline void trsm_subst64(const T* E, const T* rinv, int ri, T* xm, int si) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));   // the addresses and masks are made here, not kept from before the caller's loop
  const int i = lane & 15, g = lane >> 4;
  xm += i * si + g;
  T x[NV][4], sol[NV][4], nr[4], ec[TRSM_SG][4];
  trsm_subst_read<0>(ec, E + i);
#pragma unroll
  for (int s = 0; s < 4; s++) {
    nr[s] = -rinv[(16 * s + i) * ri];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      x[v][s] = xm[16 * s * si + 4 * v];
      sol[v][s] = T(0);
    }
  }
  trsm_subst_group<0>(x, sol, nr, ec, E + i, i);
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int v = 0; v < NV; v++) xm[16 * s * si + 4 * v] = -sol[v][s];
}

// (3) One launch solves op(A) X = B for up to TRSM_RN rows, in place: a
//     workgroup owns RB columns of B in LDS and takes the 64-row blocks in
//     dependency order.  X_b = B_b - sum_k E_bk X_k on the matrix cores (E =
//     op(A), the fragments straight from L2 as on the right side), then the
//     diagonal block by substitution, every wavefront its own vectors: backward
//     stable whatever the block's condition, and an Inf or NaN of B or A
//     reaches only the rows that depend on it, as in the reference.  All tiles
//     of the next block row are on their way from memory during a block's
//     substitution.  The bound is that chain: per block 3700 cycles of
//     substitution (58 a column), 600 to 1200 before it and about 1100 per tile
//     product.  A synchronous call with 256 x 1024 FP64 takes 45.4 us (55.0 with
//     a wavefront per vector and every tile through LDS; 49.9 with the right
//     side's inverses, which lost up to the block's condition in backward error
//     and sent an Inf or NaN to rows that do not depend on it), 8192 x 1024
//     1.93 ms (2.92, 1.86).
//     MT: the columns of M = E^T are rows of A as stored (E(i, k) = A(i, k)).
template <typename T, int RB, bool MT>
__global__ __launch_bounds__(256, 2) void trsm_left_kernel(int n, long nvec, const T* __restrict__ A, long lda,
                                                           bool lower, bool unit, T* __restrict__ B, long ldb,
                                                           const int* abort_flag) {
  constexpr int LDX = RB + 2, RT = RB / 16, NB = TRSM_NB;
  typedef MF<T> mf;
  __shared__ T Xs[TRSM_RN * LDX];   // X(k, v) at Xs[k*LDX + v]
  __shared__ T Es[NB * (NB + 1)];   // the diagonal block, an upper one reversed
  __shared__ T s_rinv[TRSM_RN];     // reciprocals of the diagonal
  if (abort_flag && *abort_flag) return;
  const long v0 = (long)blockIdx.x * RB;
  const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t >> 6);
  int lane = t & 63;
  const int nblk = (n + NB - 1) / NB;
  const int vecs = (int)min((long)RB, nvec - v0);
  auto blk_of = [&](int q) { return lower ? q : nblk - 1 - q; };   // lower: E is lower triangular
  // rows and columns past n repeat one that is there: taken out where it
  // matters.  Addresses step from load to load (a product of 64 bits each took
  // longer than the loads).
  auto fetch_diag = [&](int q, T (&f)[16]) __attribute__((always_inline)) {
    const int o = blk_of(q) * NB, c0 = min(o + w, n - 1);
    const T* src = A + (long)c0 * lda;
    const int r = min(o + lane, n - 1);
#pragma unroll
    for (int u = 0; u < 16; u++) {
      f[u] = src[r];
      src += c0 + 4 * u + 4 < n ? 4 * lda : 0;
    }
  };
  // step s of a product takes k = kof(s) + KL*(lane/16) of the tile: rows of A
  // in pieces of 128 bytes (MT), columns in pieces of 64, 16 per lane
  constexpr int V = 16 / (int)sizeof(T), KL = MT ? 1 : V;
  auto kof = [](int s) { return MT ? 4 * s : s / V * (4 * V) + s % V; };
  auto fetch = [&](int q, int p, T (&f)[16]) __attribute__((always_inline)) {
    const int i = min(blk_of(q) * NB + 16 * w + (lane & 15), n - 1), k0 = blk_of(p) * NB + KL * (lane >> 4);
    const bool whole = (blk_of(p) + 1) * NB <= n;
    if constexpr (MT) {
      const T* src = A + i + (long)min(k0, n - 1) * lda;
      if (whole) {
#pragma unroll
        for (int s = 0; s < 16; s++) {
          f[s] = *src;
          src += 4 * lda;
        }
      } else {
#pragma unroll
        for (int s = 0; s < 16; s++) {
          f[s] = *src;
          src += k0 + kof(s + 1) < n ? 4 * lda : 0;
        }
      }
    } else {
      const T* src = A + (long)i * lda;
      if (whole) {
        typedef T vec __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
#pragma unroll
        for (int s = 0; s < 16; s += V) {
          const vec x = *(const vec*)(src + k0 + kof(s));
#pragma unroll
          for (int e = 0; e < V; e++) f[s + e] = x[e];
        }
      } else {
#pragma unroll
        for (int s = 0; s < 16; s++) f[s] = src[min(k0 + kof(s), n - 1)];
      }
    }
  };
  T fd[16], f0[16], f1[16], f2[16];
  fetch_diag(0, fd);
  s_rinv[t] = t < n && !unit ? T(1) / A[t + (long)t * lda] : T(1);   // TRSM_RN threads
#pragma unroll
  for (int r0 = 0; r0 < RB; r0 += 16) {   // a thread per row of X
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = B[min(t, n - 1) + (v0 + min(r0 + u, vecs - 1)) * ldb];
#pragma unroll
    for (int u = 0; u < 16; u++) Xs[t * LDX + r0 + u] = t < n && r0 + u < vecs ? v[u] : T(0);
  }
  __syncthreads();
#pragma unroll 1
  for (int q = 0; q < nblk; q++) {
    const int b = blk_of(q);
    T* const xb = Xs + b * NB * LDX;
    asm volatile("" : "+v"(lane));   // a block's addresses are made in its turn: all kept from before the loop they spill
    const int lr = lane & 15, lg = lane >> 4;
    {
      // Of E(r, c) only r > c counts (r < c of an upper one): the other entries
      // meet rows that are solved already.  But columns past n come first in
      // an upper one and have to be zero.
      if (!lower && (b + 1) * NB > n) {
#pragma unroll
        for (int u = 0; u < 16; u++) fd[u] = b * NB + (MT ? w + 4 * u : lane) < n ? fd[u] : T(0);
      }
      const int r = MT ? lane : w, c = MT ? w : lane, dir = lower ? 1 : -1, step = dir * (MT ? 4 * (NB + 1) : 4);
      T* dst = Es + (lower ? c * (NB + 1) + r : (NB - 1 - c) * (NB + 1) + NB - 1 - r);
#pragma unroll
      for (int u = 0; u < 16; u++) {
        *dst = fd[u];
        dst += step;
      }
    }
    if (q > 0) {   // less the products of the solved blocks, in place, every wavefront its 16 rows
      typename mf::acc acc[RT];
#pragma unroll
      for (int i = 0; i < RT; i++) acc[i] = typename mf::acc{};
      auto product = [&](int p, const T (&f)[16]) __attribute__((always_inline)) {
        const T* src = Xs + (blk_of(p) * NB + KL * lg) * LDX + lr;
#pragma unroll
        for (int s = 0; s < 16; s++)
#pragma unroll
          for (int i = 0; i < RT; i++) acc[i] = mf::mma(f[s], src[kof(s) * LDX + 16 * i], acc[i]);
      };
      if (blk_of(0) == nblk - 1) {   // its rows past n
#pragma unroll
        for (int s = 0; s < 16; s++) f0[s] = (nblk - 1) * NB + KL * lg + kof(s) < n ? f0[s] : T(0);
      }
      product(0, f0);
      if (q > 1) product(1, f1);
      if (q > 2) product(2, f2);
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int x = 0; x < 4; x++) xb[(16 * w + mf::orow(lane, x)) * LDX + 16 * i + lr] -= acc[i][x];
    }
    if (q + 1 < nblk) {
      fetch_diag(q + 1, fd);
      fetch(q + 1, 0, f0);
      if (q > 0) fetch(q + 1, 1, f1);
      if (q > 1) fetch(q + 1, 2, f2);
    }
    __syncthreads();
    const int first = lower ? 0 : NB - 1, dir = lower ? 1 : -1;
    trsm_subst64<RT>(Es, s_rinv + b * NB + first, dir, xb + w * (RB / 4) + first * LDX, dir * LDX);
    __syncthreads();
  }
  int nv = vecs;
  asm volatile("" : "+s"(nv));   // nor the comparisons made for the loads
  if (t < n) {   // consecutive rows of a column of B to consecutive lanes
#pragma unroll
    for (int r = 0; r < RB; r++)
      if (r < nv) B[t + (v0 + r) * ldb] = Xs[t * LDX + r];
  }
}
static_assert(TRSM_RN == 4 * TRSM_NB, "a row per thread; at most three solved blocks before the last");

// right side: inverses of op(A)'s diagonal blocks (a0: the triangle's first
// element; the recursion splits on the 64-grid from a0)
template <typename T>
struct InvCtx {
  const T* a0 = nullptr;
  long lda = 0;
  const T* inv = nullptr;
};

template <typename T>
static void leaf(bool right, bool lower, bool trans, bool unit, long nb, long nrhs, const T* a, long lda, T* b,
                 long ldb, hipStream_t s, const int* abort_flag, const InvCtx<T>& ic) {
  if (nb <= 0 || nrhs <= 0) return;
  // 32 vectors per workgroup halve the reads of the triangle: FP32 from two
  // 16-vector workgroups per CU on (right, 16000 x 256: 54.5 us with 16 rows,
  // 49.9 with 32); FP64 is bound by its MFMAs (71.9 / 74.8)
  [[maybe_unused]] const bool wide = nrhs >= 16 * 2 * (long)rt().num_cu;
  if (right) {
    const T* inv = ic.inv + (long)(a - ic.a0) / (ic.lda + 1) / TRSM_NB * TRSM_NB * TRSM_NB;
    const bool upper = lower == trans;   // op(A)
    auto launch = [&](auto rb) {
      constexpr int RB = decltype(rb)::value;
      const unsigned g = (unsigned)((nrhs + RB - 1) / RB);
      if (trans) trsm_right_kernel<T, RB, true><<<g, 256, 0, s>>>((int)nb, nrhs, a, lda, upper, inv, b, ldb, abort_flag);
      else trsm_right_kernel<T, RB, false><<<g, 256, 0, s>>>((int)nb, nrhs, a, lda, upper, inv, b, ldb, abort_flag);
    };
    if constexpr (sizeof(T) == 4) wide ? launch(std::integral_constant<int, 32>{}) : launch(std::integral_constant<int, 16>{});
    else launch(std::integral_constant<int, 16>{});
    OBA_HIP(hipGetLastError());
    return;
  }
  const bool elower = lower != trans;   // E = op(A)
  if (nb > TRSM_NB) {
    auto launch = [&](auto rb) {
      constexpr int RB = decltype(rb)::value;
      const unsigned g = (unsigned)((nrhs + RB - 1) / RB);
      if (trans) trsm_left_kernel<T, RB, false><<<g, 256, 0, s>>>((int)nb, nrhs, a, lda, elower, unit, b, ldb, abort_flag);
      else trsm_left_kernel<T, RB, true><<<g, 256, 0, s>>>((int)nb, nrhs, a, lda, elower, unit, b, ldb, abort_flag);
    };
    if constexpr (sizeof(T) == 4) wide ? launch(std::integral_constant<int, 32>{}) : launch(std::integral_constant<int, 16>{});
    else launch(std::integral_constant<int, 16>{});
    OBA_HIP(hipGetLastError());
    return;
  }
  // a left-side triangle of one block
  trsm_leaf_kernel<T><<<(unsigned)((nrhs + 3) / 4), 256, 0, s>>>((int)nb, nrhs, a, lda, b, ldb, trans, elower, unit,
                                                                 abort_flag);
  OBA_HIP(hipGetLastError());
}

// alpha already applied; solves in place.
template <typename T>
static void rec(bool right, bool lower, bool trans, bool unit, long m, long n, const T* a, long lda, T* b,
                long ldb, hipStream_t s, const int* abort_flag, const InvCtx<T>& ic) {
  const long na = right ? n : m;   // order of the triangle
  if (na <= TRSM_RN) {   // on the 64-grid of the diagonal inverses
    leaf<T>(right, lower, trans, unit, na, right ? m : n, a, lda, b, ldb, s, abort_flag, ic);
    return;
  }
  long n1 = ((na / 2) + TRSM_NB - 1) / TRSM_NB * TRSM_NB;
  if (n1 >= na) n1 = na - TRSM_NB;
  const long n2 = na - n1;
  const T* a11 = a;
  const T* a22 = a + n1 + n1 * lda;
  const T* a21 = a + n1;          // A(n1:, :n1)
  const T* a12 = a + n1 * lda;    // A(:n1, n1:)
  const bool eff_lower = (lower != trans);  // op(A) lower triangular
  if (!right) {
    T* b1 = b;
    T* b2 = b + n1;
    if (eff_lower) {
      rec<T>(right, lower, trans, unit, n1, n, a11, lda, b1, ldb, s, abort_flag, ic);
      // B2 -= op(A)21 * X1 ; op(A)21 = A21 (lower, N) or A12^T (upper, T)
      if (!trans) gemm<T>(false, false, n2, n, n1, T(-1), a21, lda, b1, ldb, T(1), b2, ldb, s, 0, abort_flag);
      else gemm<T>(true, false, n2, n, n1, T(-1), a12, lda, b1, ldb, T(1), b2, ldb, s, 0, abort_flag);
      rec<T>(right, lower, trans, unit, n2, n, a22, lda, b2, ldb, s, abort_flag, ic);
    } else {
      rec<T>(right, lower, trans, unit, n2, n, a22, lda, b2, ldb, s, abort_flag, ic);
      // B1 -= op(A)12 * X2 ; op(A)12 = A12 (upper, N) or A21^T (lower, T)
      if (!trans) gemm<T>(false, false, n1, n, n2, T(-1), a12, lda, b2, ldb, T(1), b1, ldb, s, 0, abort_flag);
      else gemm<T>(true, false, n1, n, n2, T(-1), a21, lda, b2, ldb, T(1), b1, ldb, s, 0, abort_flag);
      rec<T>(right, lower, trans, unit, n1, n, a11, lda, b1, ldb, s, abort_flag, ic);
    }
  } else {
    T* b1 = b;
    T* b2 = b + n1 * ldb;
    if (eff_lower) {
      // X = [X1 X2], op(A) = [A11 0; op21 A22]: X2 first
      rec<T>(right, lower, trans, unit, m, n2, a22, lda, b2, ldb, s, abort_flag, ic);
      if (!trans) gemm<T>(false, false, m, n1, n2, T(-1), b2, ldb, a21, lda, T(1), b1, ldb, s, 0, abort_flag);
      else gemm<T>(false, true, m, n1, n2, T(-1), b2, ldb, a12, lda, T(1), b1, ldb, s, 0, abort_flag);
      rec<T>(right, lower, trans, unit, m, n1, a11, lda, b1, ldb, s, abort_flag, ic);
    } else {
      rec<T>(right, lower, trans, unit, m, n1, a11, lda, b1, ldb, s, abort_flag, ic);
      if (!trans) gemm<T>(false, false, m, n2, n1, T(-1), b1, ldb, a12, lda, T(1), b2, ldb, s, 0, abort_flag);
      else gemm<T>(false, true, m, n2, n1, T(-1), b1, ldb, a21, lda, T(1), b2, ldb, s, 0, abort_flag);
      rec<T>(right, lower, trans, unit, m, n2, a22, lda, b2, ldb, s, abort_flag, ic);
    }
  }
}

template <typename T>
void trsm(bool right, bool lower, bool trans, bool unit, long m, long n, T alpha, const T* a, long lda, T* b,
          long ldb, hipStream_t s, const int* abort_flag) {
  if (m <= 0 || n <= 0) return;
  if (alpha != T(1)) scale<T>(m, n, alpha, b, ldb, s);
  if (alpha == T(0)) return;
  InvCtx<T> ic;
  DevBuf invb;
  if (right) {
    // op(A) is upper when (upper, no transpose) or (lower, transpose)
    const long nblk = (n + TRSM_NB - 1) / TRSM_NB;
    invb = DevBuf(sizeof(T) * (size_t)nblk * TRSM_NB * TRSM_NB);
    trsm_inv_diag_kernel<T><<<(unsigned)nblk, 256, 0, s>>>(n, a, lda, trans, lower == trans, unit, invb.as<T>(),
                                                           abort_flag);
    OBA_HIP(hipGetLastError());
    ic.a0 = a;
    ic.lda = lda;
    ic.inv = invb.as<T>();
  }
  rec<T>(right, lower, trans, unit, m, n, a, lda, b, ldb, s, abort_flag, ic);
}

template <typename T>
size_t trsm_right_inv_bytes(long n) {
  return sizeof(T) * (size_t)((n + TRSM_NB - 1) / TRSM_NB) * TRSM_NB * TRSM_NB;
}

template <typename T>
void trsm_right_prepare(bool lower, bool trans, bool unit, long n, const T* a, long lda, T* inv, hipStream_t s) {
  if (n <= 0) return;
  const long nblk = (n + TRSM_NB - 1) / TRSM_NB;
  trsm_inv_diag_kernel<T><<<(unsigned)nblk, 256, 0, s>>>(n, a, lda, trans, lower == trans, unit, inv, nullptr);
  OBA_HIP(hipGetLastError());
}

template <typename T>
void trsm_right_prepared(bool lower, bool trans, bool unit, long m, long n, const T* a, long lda, T* b, long ldb,
                         const T* inv, hipStream_t s, const int* abort_flag) {
  if (m <= 0 || n <= 0) return;
  InvCtx<T> ic;
  ic.a0 = a;
  ic.lda = lda;
  ic.inv = inv;
  rec<T>(true, lower, trans, unit, m, n, a, lda, b, ldb, s, abort_flag, ic);
}

template size_t trsm_right_inv_bytes<double>(long);
template size_t trsm_right_inv_bytes<float>(long);
template void trsm_right_prepare<double>(bool, bool, bool, long, const double*, long, double*, hipStream_t);
template void trsm_right_prepare<float>(bool, bool, bool, long, const float*, long, float*, hipStream_t);
template void trsm_right_prepared<double>(bool, bool, bool, long, long, const double*, long, double*, long,
                                          const double*, hipStream_t, const int*);
template void trsm_right_prepared<float>(bool, bool, bool, long, long, const float*, long, float*, long,
                                         const float*, hipStream_t, const int*);
template void trsm<double>(bool, bool, bool, bool, long, long, double, const double*, long, double*, long, hipStream_t, const int*);
template void trsm<float>(bool, bool, bool, bool, long, long, float, const float*, long, float*, long, hipStream_t, const int*);

}  // namespace oba
