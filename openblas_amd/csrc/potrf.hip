// Cholesky factorization (potrf, lower and upper), device pointers.
//
// Reference semantics (lapack/potf2/potf2_L.c:50-97, potrf_L_single.c:81-236,
// potrf_U_single.c:79-193): only the selected triangle is read or written;
// at column j, ajj = a_jj - sum_k l_jk^2; if ajj <= 0 the value is stored in
// a_jj and the routine returns info = j+1 without touching later columns
// (a NaN ajj is not caught, exactly like the reference's `ajj <= 0` test);
// otherwise a_jj = sqrt(ajj) and the column below is scaled by 1/a_jj.
//
// MI355X design: recursion on halves (64-column grid): L21 <- A21*L11^-T is a
// right-side TRSM, A22 -= L21*L21^T is an MFMA GEMM restricted to the lower
// triangle (the role of the reference's SYRK kernel); 64x64 diagonal leaves
// are factored and inverted by one workgroup.  Large lower
// factorizations run blocked with look-ahead (potrf_blocked).  A failing leaf raises a device flag
// that turns every later kernel of the same call into a no-op, so the call
// stops where the reference stops without a host round trip per leaf.
#include "kernels.h"
#include "tri_inv.h"
#include <cmath>

namespace oba {

constexpr int PO_NB = 64;

__device__ inline float po_rl(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ inline double po_rl(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// Factor the nb x nb (nb <= 64) diagonal block at a (lower: E(i,k) =
// a[i + k*lda]; upper: E(i,k) = a[k + i*lda], i >= k) and, when inv is not
// null, invert the factor for the right-side solve that follows
// (M = L^T: M^{-1}(i,j) = L^{-1}(j,i) at inv[i*64 + j], as
// trsm_inv_diag_kernel leaves it); info and the failure flag take the global
// column offset j0.
//
// The bound is the chain of 64 columns (diagonal, square root, reciprocal,
// multipliers, next column).  The block sits in LDS and is taken in four
// steps of 16 columns: wavefront 0 factors a step with row i in lane i and the
// 16 columns in registers, every value another row needs read with
// v_readlane (no LDS, no barrier inside a step); then all four wavefronts
// subtract the step's products from the later columns, 16x16 tiles on the
// matrix cores; wavefronts 1 to 3 invert the finished 16x16 diagonal blocks
// and join the inverse 16 -> 32 -> 64 by small MFMA products while wavefront 0
// factors the next step.  22 us FP64 and 16 FP32 with the inverse.  One wavefront
// with all 64 columns in registers, every column updating all later ones with
// multipliers read back from LDS, took 62 and 50 us per leaf, and the
// inversion was a launch of its own (16 and 14 us).
//
// Column j: ajj <= 0 (not NaN) is stored as it is and stops the leaf
// (potf2_L.c:71-75); otherwise the column is scaled by 1/l_jj (its SCAL_K).
// Rows and columns past nb hold the identity.
template <typename T>
__global__ __launch_bounds__(256) void potrf_leaf_kernel(int nb, T* a, long lda, bool upper, long j0, int* info,
                                                         T* inv) {
  constexpr int NB = PO_NB, LD = NB + 1;
  typedef MF<T> mf;
  __shared__ T S[NB * LD];   // E(i, c) at S[c*LD + i]
  __shared__ T Y[NB * LD];   // L^{-1}(i, c) at Y[c*LD + i]
  __shared__ T U[NB * LD];   // products of the joins
  __shared__ T s_rinv[NB];
  __shared__ int s_fail;
  if (*info) return;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), lr = lane & 15, lg = lane >> 4;
  {
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int f = (t + 256 * u) & 63, g = (t + 256 * u) >> 6;   // f contiguous in memory
      v[u] = a[min(f, nb - 1) + (long)min(g, nb - 1) * lda];
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int f = (t + 256 * u) & 63, g = (t + 256 * u) >> 6, i = upper ? g : f, c = upper ? f : g;
      S[c * LD + i] = i >= c && i < nb && c < nb ? v[u] : (i == c ? T(1) : T(0));
      Y[c * LD + i] = T(0);
    }
  }
  if (t == 0) s_fail = 0;
  __syncthreads();
  int fail = 0;
#pragma unroll 1
  for (int q = 0; q < 5; q++) {
    if (w == 0 && q < 4) {
      // row (lane + 16q) mod 64 in this lane: the step's own 16 rows are in
      // lanes 0..15 whatever q is, so every v_readlane has a constant lane
      // (with a lane index from an SGPR they took 25 cycles each, 740 a column)
      const int row = (lane + 16 * q) & 63;
      const bool below = lane < 64 - 16 * q;   // rows 16q and later
      T x[16];
#pragma unroll
      for (int k = 0; k < 16; k++) x[k] = S[(16 * q + k) * LD + row];
      // no branch inside the step: the tail of a column's update runs beside
      // the next column's square root and reciprocal
      bool low = false;
      T rv = T(0);
#pragma unroll
      for (int jj = 0; jj < 16; jj++) {
        const T d = po_rl(x[jj], jj);
        low |= d <= T(0);
        const T ljj = sqrt(d);
        const T rinv = T(1) / ljj;
        const T li = x[jj] * rinv;
#pragma unroll
        for (int k = jj + 1; k < 16; k++) x[k] -= li * po_rl(li, k);
        x[jj] = lane == jj ? ljj : li;
        rv = lane == jj ? rinv : rv;
      }
      int bad = 0;
      if (low) {   // the step again, up to the diagonal that is stored as it is
#pragma unroll
        for (int k = 0; k < 16; k++) x[k] = S[(16 * q + k) * LD + row];
#pragma unroll
        for (int jj = 0; jj < 16; jj++) {
          const T d = po_rl(x[jj], jj);
          if (!bad && d <= T(0)) bad = 16 * q + jj + 1;
          if (bad) continue;
          const T ljj = sqrt(d);
          const T li = x[jj] * (T(1) / ljj);
#pragma unroll
          for (int k = jj + 1; k < 16; k++) x[k] -= li * po_rl(li, k);
          x[jj] = lane == jj ? ljj : li;
        }
      }
      if (lane < 16) s_rinv[16 * q + lane] = rv;
      if (below) {
#pragma unroll
        for (int k = 0; k < 16; k++)
          if (lane >= k) S[(16 * q + k) * LD + row] = x[k];
      }
      if (lane == 0 && bad) s_fail = bad;
    }
    if (inv) {   // beside the factorization of a step: the inverse, as far as the columns are final
      if (w == 3 && q > 0) {
        tri_inv16(S, Y, s_rinv, 16 * (q - 1));
        if (!(q & 1)) {   // join with the block before
          wave_fence();
          tri_prod<1>(U, S, Y, q - 1, q - 2, q - 2, T(1));
          wave_fence();
          tri_prod<1>(Y, Y, U, q - 1, q - 2, q - 1, T(-1));
        }
      }
      if (q == 3 && (w == 1 || w == 2)) {   // L21 Y11
#pragma unroll 1
        for (int u = 0; u < 2; u++) tri_prod<2>(U, S, Y, 1 + w, u, 0, T(1));
      }
    }
    if (q == 4) break;
    __syncthreads();
    fail = __builtin_amdgcn_readfirstlane(s_fail);
    if (fail) break;
    // the step's products leave the later columns, one tile per wavefront at
    // a time: (1,1) (2,1) (2,2) (3,1) (3,2) (3,3), offset by q
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int tile = w + 4 * u, ti = tile < 1 ? 1 : tile < 3 ? 2 : 3, tj = tile - ti * (ti - 1) / 2 + 1;
      const int ri = q + ti, ci = q + tj;
      if (tile < 6 && ri < 4) {
        const T* l = S + (16 * q + lg) * LD;
        typename mf::acc acc{};
#pragma unroll
        for (int s = 0; s < 4; s++)
          acc = mf::mma(l[4 * s * LD + 16 * ci + lr], l[4 * s * LD + 16 * ri + lr], acc);
#pragma unroll
        for (int r = 0; r < 4; r++) S[(16 * ci + mf::orow(lane, r)) * LD + 16 * ri + lr] -= acc[r];
      }
    }
    __syncthreads();
  }
  // the factor back to memory (a failed leaf: the columns before the failing
  // one, and its diagonal)
  const int cols = fail ? fail - 1 : nb;
#pragma unroll
  for (int u = 0; u < 16; u++) {
    const int f = (t + 256 * u) & 63, g = (t + 256 * u) >> 6, i = upper ? g : f, c = upper ? f : g;
    if (i < nb && i >= c && (c < cols || (c == cols && i == c && c < nb))) a[f + (long)g * lda] = S[c * LD + i];
  }
  if (fail) {
    if (t == 0) *info = (int)(j0 + fail);
    return;
  }
  if (!inv) return;
  __syncthreads();
  tri_prod<2>(Y, Y, U, 2 + (w >> 1), w & 1, 2, T(-1));   // Y21 = -Y22 (L21 Y11)
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 16; u++) {
    const int idx = t + 256 * u, i = idx >> 6, j = idx & 63;
    inv[idx] = i < nb && j < nb ? Y[i * LD + j] : T(0);
  }
}

// inv (lower): the inverses of the 64x64 diagonal blocks, block b of the
// matrix at inv + b*64*64, left by the leaves for the right-side solves
template <typename T>
static void potrf_rec(bool lower, long j0, long nc, T* a, long lda, int* info, T* inv, hipStream_t s) {
  T* a11 = a + j0 + j0 * lda;
  T* inv11 = inv ? inv + j0 * PO_NB : nullptr;   // j0 is a multiple of 64
  if (nc <= PO_NB) {
    potrf_leaf_kernel<T><<<1, 256, 0, s>>>((int)nc, a11, lda, !lower, j0, info, inv11);
    OBA_HIP(hipGetLastError());
    return;
  }
  long n1 = ((nc / 2) + PO_NB - 1) / PO_NB * PO_NB;
  if (n1 >= nc) n1 = nc - PO_NB;
  const long n2 = nc - n1;
  potrf_rec<T>(lower, j0, n1, a, lda, info, inv, s);
  T* a22 = a + (j0 + n1) + (j0 + n1) * lda;
  if (lower) {
    T* a21 = a + (j0 + n1) + j0 * lda;
    trsm_right_prepared<T>(true, true, false, n2, n1, a11, lda, a21, lda, inv11, s, info);   // A21 L11^-T
    gemm<T>(false, true, n2, n2, n1, T(-1), a21, lda, a21, lda, T(1), a22, lda, s, 1, info);
  } else {
    T* a12 = a + j0 + (j0 + n1) * lda;
    trsm<T>(false, false, true, false, n1, n2, T(1), a11, lda, a12, lda, s, info);  // U11^-T A12
    gemm<T>(true, false, n2, n2, n1, T(-1), a12, lda, a12, lda, T(1), a22, lda, s, 2, info);
  }
  potrf_rec<T>(lower, j0 + n1, n2, a, lda, info, inv, s);
}

// Blocked right-looking Cholesky (lower) with look-ahead, for large n, as
// the blocked LU: the columns are cut into blocks of nb.  On the caller's
// stream: block k's diagonal block (the recursion above), then the rows of
// its panel that belong to block k+1 (right-side TRSM with the 64x64
// diagonal inverses computed once) and block k+1's diagonal update; block
// k+1 is factored next.  Meanwhile the bulk stream (CU mask, all but the
// reserved CUs) solves the rest of the panel and updates the trailing
// matrix (one GEMM for block k+1's column below its diagonal block, one
// lower-restricted GEMM for the rest), and the caller's stream waits for it
// before it touches those rows.  Every kernel takes the failure flag: after
// a non-positive pivot the rest of the call is a no-op, as in the
// recursion.  The trailing sums run over blocks instead of recursion
// halves: a different association of the same products.
template <typename T>
static void potrf_blocked(long n, T* a, long lda, int* info, long nb, T* inv, hipStream_t s) {
  Runtime& r = rt();
  hipStream_t M = s, X = bulk_stream();
  auto at = [&](long i, long j) { return a + i + j * lda; };
  potrf_rec<T>(true, 0, std::min(nb, n), a, lda, info, inv, M);
  bool pending = false;
  for (long jb = 0; jb < n; jb += nb) {
    const long w = std::min(nb, n - jb), jn = jb + w;
    if (pending) {   // the trailing update by the previous block has finished
      OBA_HIP(hipStreamWaitEvent(M, r.ev_b, 0));
      pending = false;
    }
    if (jn >= n) break;
    const long w1 = std::min(nb, n - jn);
    const T* l11 = at(jb, jb);
    const T* inv11 = inv + jb * PO_NB;
    trsm_right_prepared<T>(true, true, false, w1, w, l11, lda, at(jn, jb), lda, inv11, M, info);
    gemm<T>(false, true, w1, w1, w, T(-1), at(jn, jb), lda, at(jn, jb), lda, T(1), at(jn, jn), lda, M, 1, info);
    const long rest = n - (jn + w1);
    if (rest > 0) {
      OBA_HIP(hipEventRecord(r.ev_a, M));
      OBA_HIP(hipStreamWaitEvent(X, r.ev_a, 0));
      trsm_right_prepared<T>(true, true, false, rest, w, l11, lda, at(jn + w1, jb), lda, inv11, X, info);
      gemm<T>(false, true, rest, w1, w, T(-1), at(jn + w1, jb), lda, at(jn, jb), lda, T(1), at(jn + w1, jn), lda, X, 0,
              info);
      gemm<T>(false, true, rest, rest, w, T(-1), at(jn + w1, jb), lda, at(jn + w1, jb), lda, T(1),
              at(jn + w1, jn + w1), lda, X, 1, info);
      OBA_HIP(hipEventRecord(r.ev_b, X));
      pending = true;
    }
    potrf_rec<T>(true, jn, w1, a, lda, info, inv, M);
  }
  if (pending) OBA_HIP(hipStreamWaitEvent(M, r.ev_b, 0));
}

// block width of the look-ahead driver (OPENBLAS_AMD_PO_NB; 0 turns it off);
// it is used from 4 blocks on
template <typename T>
static long potrf_block_nb(long n) {
  // swept with the 64x64 leaves inverted in place, ms for widths 256 / 384 /
  // 512 / 640: dpotrf n = 5000 3.54 / 3.86 / 3.71 / 3.99, 8192 7.25 / 7.43 /
  // 7.28 / 7.70, 16384 35.0 / 34.3 / 33.0 / 33.5; spotrf 8192 5.37 / 5.39 /
  // 5.48 / 5.77, 16384 21.2 / 20.4 / 19.8 / 20.3: short chains favour the
  // narrow block, large trailing updates the deeper K
  long v = n >= 12288 ? 512 : 256;
  if (const char* e = getenv("OPENBLAS_AMD_PO_NB")) v = atol(e);
  return v;
}

template <typename T>
int potrf(bool lower, long n, T* a, long lda, hipStream_t s) {
  if (n <= 0) return 0;
  DevBuf ib(sizeof(int) * 64);
  int* info = ib.as<int>();
  OBA_HIP(hipMemsetAsync(info, 0, sizeof(int), s));
  const long nb = potrf_block_nb<T>(n);
  const bool blocked = lower && nb >= PO_NB && nb % PO_NB == 0 && n >= 4 * nb;
  DevBuf invb(lower ? trsm_right_inv_bytes<T>(n) : 0);
  if (blocked) {
    invb.use_on(bulk_stream());   // read by the bulk stream's solves
    potrf_blocked<T>(n, a, lda, info, nb, invb.as<T>(), s);
  } else {
    potrf_rec<T>(lower, 0, n, a, lda, info, invb.as<T>(), s);
  }
  int h = 0;
  OBA_HIP(hipMemcpyAsync(&h, info, sizeof(int), hipMemcpyDeviceToHost, s));
  OBA_HIP(hipStreamSynchronize(s));
  return h;
}

template int potrf<double>(bool, long, double*, long, hipStream_t);
template int potrf<float>(bool, long, float*, long, hipStream_t);

}  // namespace oba
