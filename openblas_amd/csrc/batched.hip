// Batched small problems (GEMM, LU, LU solve, Cholesky) in one persistent
// launch per kind.  The reference has a batched GEMM only
// (interface/gemm_batch.c:117, one problem per thread in
// driver/level3/gemm_batch_thread.c:79); batched getrf/getrs/potrf have no
// reference entry point and follow the single-problem semantics of
// lapack/getf2/getf2_k.c, lapack/getrs/getrs_single.c and
// lapack/potf2/potf2_L.c problem by problem.
//
// MI355X design:
//  * a problem table (BDesc) sorted largest-first lives in HBM; workgroups
//    (GEMM tiles, LU, Cholesky) or wavefronts (solves) pull the next item
//    from an atomic queue, so 10^4 uneven problems keep all 256 CUs busy
//    without one launch per problem;
//  * GEMM: 64- and 32-wide output tiles with the single GEMM's loads and main
//    loop, one queue per XCD;
//  * LU (m <= 512): batched_lu.h, a launch per size class where the classes fill
//    the device;
//  * Cholesky (n <= 512): same row-owner panel, one barrier per column,
//    SYRK-shaped trailing update of the lower triangle;
//  * LU solve (n <= 512): one wavefront per problem, the right-hand side in
//    registers (lane l owns rows l, l+64, ...), row interchanges by lane
//    reads/writes, triangular sweeps with 8 columns of the factor loaded
//    per step;
//  * the launch sequence (queue reset by a fill kernel, the kernel) is
//    captured once in a hipGraph per problem table and replayed while the
//    table is unchanged; tile width, panel width and persistent grid size
//    are chosen per batch shape by timing the candidates on scratch copies.
#include "batched.h"
#include "kernels.h"
#include "lu_device.h"
#include "lu_internal.h"
#include "gemm_tile.h"
#include <algorithm>
#include <climits>
#include <cstring>
#include <map>
#include <string>
#include <type_traits>
#include <vector>

namespace oba {

// The problems' pointers come from the descriptor table, so the compiler
// sees generic pointers and emits flat loads and stores, which also count
// against the LDS wait counter: every LDS wait then waits for outstanding
// memory operations too.  They point to device memory: use them as global.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;

}  // namespace oba

#include "batched_gemm.h"
#include "batched_lu.h"

namespace oba {

// ---- small device helpers ----------------------------------------------------
__device__ inline double bcast_lane(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}
__device__ inline float bcast_lane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline int bcast_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

template <typename T>
__device__ inline T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

__global__ void bzero_kernel(unsigned* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// copies operand a or b of every problem from src to dst descriptors (rows x
// cols, each with its own leading dimension): scratch copies of in/out operands
// for the tuner
template <typename T>
__global__ void bcopy_kernel(const BDesc* __restrict__ src, const BDesc* __restrict__ dst, bool b_operand, int rows_field,
                             int cols_field) {
  const BDesc& s = src[blockIdx.y];
  const BDesc& d = dst[blockIdx.y];
  const int* fs = &s.m;
  const long rows = fs[rows_field], cols = fs[cols_field];
  const long lds = b_operand ? s.ldb : s.lda, ldd = b_operand ? d.ldb : d.lda;
  gptr<const T> a = (gptr<const T>)(b_operand ? s.b : s.a);
  gptr<T> b = (gptr<T>)(b_operand ? d.b : d.a);
  const long total = rows * cols;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const long i = e % rows, j = e / rows;
    b[i + j * ldd] = a[i + j * lds];
  }
}

// ---- batched Cholesky (n <= 256*RPT) -------------------------------------------
// LOWER: A = L*L^T with L(i,c) = a[i + c*lda]; upper: A = U^T*U, U = L^T,
// L(i,c) = a[c + i*lda].  Failure rule of lapack/potf2/potf2_L.c:71-75: an
// updated diagonal <= 0 is stored and info = j+1; NaN passes through.
template <typename T, int RPT, int W, bool LOWER>
__global__ __launch_bounds__(256) void bpotrf_kernel(const BDesc* __restrict__ desc, int count,
                                                     unsigned* __restrict__ counter, int* __restrict__ info_out) {
  constexpr int NT = 256, UB = NT, LDL = W + 1, BU = RPT == 1 ? 32 : 16;
  typedef typename RowVec<T, W>::type RV;
  __shared__ T s_col[2][W];
  __shared__ T s_l[UB * LDL];
  __shared__ int s_item[2];
  const int t = threadIdx.x;

  if (t == 0) s_item[0] = (int)atomicAdd(counter, 1u);
  __syncthreads();
  int cur = 0;
  int it = s_item[0];
  while (it < count) {
    if (t == 0) s_item[cur ^ 1] = (int)atomicAdd(counter, 1u);
    const BDesc& d = desc[it];
    const int n = d.n;
    const long lda = d.lda;
    gptr<T> A = (gptr<T>)d.a;
    auto at = [&](long i, long c) -> decltype(A[0])& { return LOWER ? A[i + c * lda] : A[c + i * lda]; };
    int info = 0;
    #pragma unroll 1
    for (int j0 = 0; j0 < n; j0 += W) {
      const int w = min(W, n - j0);
      RV x[RPT];
      int row[RPT];
      bool live[RPT];
#pragma unroll
      for (int q = 0; q < RPT; q++) {
        row[q] = j0 + t + NT * q;
        live[q] = row[q] < n;
#pragma unroll
        for (int c = 0; c < W; c++) x[q][c] = (live[q] && c < w && j0 + c <= row[q]) ? at(row[q], j0 + c) : T(0);
      }
      int fail = 0;
      #pragma unroll 1
      for (int k = 0; k < w; k++) {
        const int j = j0 + k, buf = k & 1;
#pragma unroll
        for (int q = 0; q < RPT; q++)
          if (live[q] && row[q] >= j && row[q] < j0 + w) s_col[buf][row[q] - j0] = pick<RV, W>(x[q], k);
        __syncthreads();
        const T dj = s_col[buf][k];
        if (dj <= T(0)) {   // uniform: every thread read the same value
#pragma unroll
          for (int q = 0; q < RPT; q++)
            if (live[q] && row[q] == j) at(j, j) = dj;
          fail = j + 1;
          break;
        }
        const T sj = sqrt(dj);
        const T rinv = T(1) / sj;
#pragma unroll
        for (int q = 0; q < RPT; q++) {
          if (!live[q] || row[q] < j) continue;
          if (row[q] == j) {
#pragma unroll
            for (int c = 0; c < W; c++)
              if (c == k) x[q][c] = sj;
          } else {
            const T l = pick<RV, W>(x[q], k) * rinv;
#pragma unroll
            for (int c = 0; c < W; c++) {
              if (c == k) x[q][c] = l;
              else if (c > k && c < w && j0 + c <= row[q]) x[q][c] -= l * (s_col[buf][c] * rinv);
            }
          }
        }
      }
      const int kdone = fail ? fail - 1 - j0 : w;
#pragma unroll
      for (int q = 0; q < RPT; q++) {
        if (!live[q]) continue;
#pragma unroll
        for (int c = 0; c < W; c++)
          if (c < kdone && j0 + c <= row[q]) at(row[q], j0 + c) = x[q][c];
      }
      if (fail) { info = fail; break; }
      if constexpr (RPT == 1) {
        // trailing SYRK A22 -= L21 L21^T on MFMA 16x16 tiles of the lower
        // triangle (4 wavefronts, GT tiles each per step, their C elements
        // loaded before the products so one memory latency covers GT tiles)
        typedef MF<T> mf;
        const int c0 = j0 + w, nr = n - c0;
        if (nr > 0) {
          if (live[0] && row[0] >= c0) {
#pragma unroll
            for (int c = 0; c < W; c++) s_l[(row[0] - c0) * LDL + c] = c < w ? x[0][c] : T(0);
          }
          __syncthreads();
          const int lane = t & 63, wave = t >> 6;
          const int nt = (nr + 15) / 16, ntiles = nt * (nt + 1) / 2;
          constexpr int GT = 4;
          #pragma unroll 1
          for (int tb = wave * GT; tb < ntiles; tb += 4 * GT) {
            int ti[GT], tj[GT];
            T cv[GT][4];
            typename mf::acc acc[GT];
#pragma unroll
            for (int g = 0; g < GT; g++) {
              const int tile = min(tb + g, ntiles - 1);
              int a0 = (int)((sqrtf(8.0f * (float)tile + 1.0f) - 1.0f) * 0.5f);
              while (a0 * (a0 + 1) / 2 > tile) a0--;
              while ((a0 + 1) * (a0 + 2) / 2 <= tile) a0++;
              ti[g] = a0;
              tj[g] = tile - a0 * (a0 + 1) / 2;
#pragma unroll
              for (int r = 0; r < 4; r++) {
                const int ri = c0 + ti[g] * 16 + (lane & 15), cj = c0 + tj[g] * 16 + mf::orow(lane, r);
                cv[g][r] = (tb + g < ntiles && ri < n && ri >= cj) ? at(ri, cj) : T(0);
              }
            }
#pragma unroll
            for (int g = 0; g < GT; g++) {
              acc[g] = typename mf::acc{T(0), T(0), T(0), T(0)};
              const int ra = ti[g] * 16 + (lane & 15), rb = tj[g] * 16 + (lane & 15);
#pragma unroll
              for (int kk = 0; kk < W; kk += 4) {
                const int k = kk + (lane >> 4);
                const T fa = ra < nr ? s_l[ra * LDL + k] : T(0);
                const T fb = rb < nr ? s_l[rb * LDL + k] : T(0);
                acc[g] = mf::mma(fb, fa, acc[g]);
              }
            }
#pragma unroll
            for (int g = 0; g < GT; g++)
#pragma unroll
              for (int r = 0; r < 4; r++) {
                const int ri = c0 + ti[g] * 16 + (lane & 15), cj = c0 + tj[g] * 16 + mf::orow(lane, r);
                if (tb + g < ntiles && ri < n && ri >= cj) at(ri, cj) = cv[g][r] - acc[g][r];
              }
          }
        }
      } else {
      #pragma unroll 1
      for (int c0 = j0 + w; c0 < n; c0 += UB) {
#pragma unroll
        for (int q = 0; q < RPT; q++)
          if (live[q] && row[q] >= c0 && row[q] < c0 + UB) {
#pragma unroll
            for (int c = 0; c < W; c++)
              if (c < w) s_l[(row[q] - c0) * LDL + c] = x[q][c];
          }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RPT; q++) {
          if (!live[q] || row[q] < c0) continue;
          const int cend = min(row[q], c0 + UB - 1);
          // BU columns per step, their loads issued together
          #pragma unroll 1
          for (int cb = c0; cb <= cend; cb += BU) {
            T a[BU];
#pragma unroll
            for (int u = 0; u < BU; u++) a[u] = cb + u <= cend ? at(row[q], cb + u) : T(0);
#pragma unroll
            for (int u = 0; u < BU; u++) {
              if (cb + u <= cend) {
                const T* lr = s_l + (cb + u - c0) * LDL;
                T v = a[u];
#pragma unroll
                for (int k = 0; k < W; k++)
                  if (k < w) v -= x[q][k] * lr[k];
                at(row[q], cb + u) = v;
              }
            }
          }
        }
        __syncthreads();
      }
      }
      __syncthreads();
    }
    if (t == 0) info_out[it] = info;
    __syncthreads();
    cur ^= 1;
    it = s_item[cur];
  }
}

// ---- batched LU solve (n <= 64*S), one wavefront per problem -------------------
// x <- A^-1 b (TRANS: A^-T b) with the factors and pivots of getrf, as
// lapack/getrs/getrs_single.c: interchanges, unit-L sweep, U sweep (or the
// transposed sweeps and the interchanges in reverse).  Lane l owns rows
// l + 64s of the right-hand side; slot indices s are compile-time constants
// (static_for) so x stays in registers.
template <int I, int N, typename F>
__device__ __attribute__((always_inline)) inline void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

template <typename T, int S>
__device__ __attribute__((always_inline)) inline void lane_swap(T (&x)[S], int s, int l, int p) {
  const int ps = p >> 6, pl = p & 63, lane = threadIdx.x & 63;
  T a = x[0], src = x[0];
#pragma unroll
  for (int s2 = 1; s2 < S; s2++) {
    a = (s == s2) ? x[s2] : a;
    src = (ps == s2) ? x[s2] : src;
  }
  const T va = bcast_lane(a, l);
  const T vb = bcast_lane(src, pl);
#pragma unroll
  for (int s2 = 0; s2 < S; s2++) {
    if (s2 == s) x[s2] = (lane == l) ? vb : x[s2];
    if (s2 == ps) x[s2] = (lane == pl) ? va : x[s2];
  }
}

template <typename T, int S, bool TRANS>
__global__ __launch_bounds__(256) void bgetrs_kernel(const BDesc* __restrict__ desc, int count,
                                                     unsigned* __restrict__ counter) {
  constexpr int U = 8;   // factor columns loaded per step
  const int lane = threadIdx.x & 63;
  int it = 0;
  if (lane == 0) it = (int)atomicAdd(counter, 1u);
  it = __builtin_amdgcn_readfirstlane(__shfl(it, 0));
  while (it < count) {
    int nx = 0;
    if (lane == 0) nx = (int)atomicAdd(counter, 1u);
    const BDesc& d = desc[it];
    const int n = d.n, nrhs = d.k;
    const long lda = d.lda, ldb = d.ldb;
    gptr<const T> A = (gptr<const T>)d.a;
    gptr<T> B = (gptr<T>)d.b;
    int ip[S];
#pragma unroll
    for (int s = 0; s < S; s++) {
      const int i = 64 * s + lane;
      ip[s] = i < n ? ((gptr<const int>)d.ipiv)[i] - 1 : i;
    }
#pragma unroll 1
    for (int r = 0; r < nrhs; r++) {
      auto b = B + r * ldb;
      T x[S];
#pragma unroll
      for (int s = 0; s < S; s++) {
        const int i = 64 * s + lane;
        x[s] = i < n ? b[i] : T(0);
      }
      // interchanges k = 0 .. n-1 (forward) or n-1 .. 0 (TRANS, after the sweeps)
      auto swaps = [&](bool forward) __attribute__((always_inline)) {
#pragma unroll 1
        for (int kk = 0; kk < n; kk++) {
          const int k = forward ? kk : n - 1 - kk;
          const int s = k >> 6, l = k & 63;
          int pv = ip[0];
#pragma unroll
          for (int s2 = 1; s2 < S; s2++) pv = (s == s2) ? ip[s2] : pv;
          const int p = bcast_lane(pv, l);
          if (p != k) lane_swap<T, S>(x, s, l, p);
        }
      };
      if (!TRANS) {
        swaps(true);
        // unit lower sweep: x_i -= L(i,k) x_k for i > k
        static_for<0, S>([&](auto sc) __attribute__((always_inline)) {
          constexpr int s = decltype(sc)::value;
#pragma unroll 1
          for (int l0 = 0; l0 < 64 && 64 * s + l0 < n; l0 += U) {
            T cv[U][S];
#pragma unroll
            for (int e = 0; e < U; e++) {
              const int k = 64 * s + l0 + e;
#pragma unroll
              for (int s2 = s; s2 < S; s2++) {
                const int i = 64 * s2 + lane;
                cv[e][s2] = (k < n && i > k && i < n) ? A[i + k * lda] : T(0);
              }
            }
#pragma unroll
            for (int e = 0; e < U; e++) {
              const int k = 64 * s + l0 + e;
              if (k < n) {
                const T xk = bcast_lane(x[s], l0 + e);
#pragma unroll
                for (int s2 = s; s2 < S; s2++)
                  if (64 * s2 + lane > k) x[s2] -= cv[e][s2] * xk;
              }
            }
          }
        });
        // upper sweep, k = n-1 .. 0: x_k /= U(k,k); x_i -= U(i,k) x_k for i < k
        static_for<0, S>([&](auto sc) __attribute__((always_inline)) {
          constexpr int s = S - 1 - decltype(sc)::value;
#pragma unroll 1
          for (int l0 = 64 - U; l0 >= 0; l0 -= U) {
            if (64 * s + l0 >= n) continue;
            T cv[U][S];
#pragma unroll
            for (int e = 0; e < U; e++) {
              const int k = 64 * s + l0 + e;
#pragma unroll
              for (int s2 = 0; s2 <= s; s2++) {
                const int i = 64 * s2 + lane;
                cv[e][s2] = (k < n && i <= k) ? A[i + k * lda] : T(0);
              }
            }
#pragma unroll
            for (int e = U - 1; e >= 0; e--) {
              const int k = 64 * s + l0 + e;
              if (k < n) {
                x[s] = (lane == l0 + e) ? x[s] / cv[e][s] : x[s];
                const T xk = bcast_lane(x[s], l0 + e);
#pragma unroll
                for (int s2 = 0; s2 <= s; s2++)
                  if (64 * s2 + lane < k) x[s2] -= cv[e][s2] * xk;
              }
            }
          }
        });
      } else {
        // U^T sweep, i = 0 .. n-1: x_i = (x_i - sum_{k<i} U(k,i) x_k) / U(i,i)
        static_for<0, S>([&](auto sc) __attribute__((always_inline)) {
          constexpr int s = decltype(sc)::value;
#pragma unroll 1
          for (int l0 = 0; l0 < 64 && 64 * s + l0 < n; l0 += U) {
            T cv[U][S];
#pragma unroll
            for (int e = 0; e < U; e++) {
              const int i = 64 * s + l0 + e;
#pragma unroll
              for (int s2 = 0; s2 <= s; s2++) {
                const int k = 64 * s2 + lane;
                cv[e][s2] = (i < n && k <= i) ? A[k + i * lda] : T(0);
              }
            }
#pragma unroll
            for (int e = 0; e < U; e++) {
              const int i = 64 * s + l0 + e;
              if (i < n) {
                T part = T(0);
#pragma unroll
                for (int s2 = 0; s2 <= s; s2++)
                  if (64 * s2 + lane < i) part += cv[e][s2] * x[s2];
                const T sum = wave_sum(part);
                const T dia = bcast_lane(cv[e][s], l0 + e);
                x[s] = (lane == l0 + e) ? (x[s] - sum) / dia : x[s];
              }
            }
          }
        });
        // L^T sweep (unit), i = n-1 .. 0: x_i -= sum_{k>i} L(k,i) x_k
        static_for<0, S>([&](auto sc) __attribute__((always_inline)) {
          constexpr int s = S - 1 - decltype(sc)::value;
#pragma unroll 1
          for (int l0 = 64 - U; l0 >= 0; l0 -= U) {
            if (64 * s + l0 >= n) continue;
            T cv[U][S];
#pragma unroll
            for (int e = 0; e < U; e++) {
              const int i = 64 * s + l0 + e;
#pragma unroll
              for (int s2 = s; s2 < S; s2++) {
                const int k = 64 * s2 + lane;
                cv[e][s2] = (i < n && k > i && k < n) ? A[k + i * lda] : T(0);
              }
            }
#pragma unroll
            for (int e = U - 1; e >= 0; e--) {
              const int i = 64 * s + l0 + e;
              if (i < n) {
                T part = T(0);
#pragma unroll
                for (int s2 = s; s2 < S; s2++)
                  if (64 * s2 + lane > i && 64 * s2 + lane < n) part += cv[e][s2] * x[s2];
                const T sum = wave_sum(part);
                x[s] = (lane == l0 + e) ? x[s] - sum : x[s];
              }
            }
          }
        });
        swaps(false);
      }
#pragma unroll
      for (int s = 0; s < S; s++) {
        const int i = 64 * s + lane;
        if (i < n) b[i] = x[s];
      }
    }
    it = __builtin_amdgcn_readfirstlane(__shfl(nx, 0));
  }
}

// ---- host side: plans, graphs, tuning -------------------------------------------
namespace {

constexpr int BCTR = 8 * BG_CTR;   // words of a plan's queue counters

struct Cfg {
  int var = 0;    // kernel variant
  int grid = 2;   // persistent workgroups per CU
};

struct Plan {
  Cfg cfg;
  std::vector<char> ctx;
  std::vector<BDesc> probs;   // the table on the device; empty: none
  DevBuf tab;       // BDesc table (+ GEMM work list)
  DevBuf ctr;       // queue counter
  DevBuf info;      // per-problem info
  hipGraphExec_t exec = nullptr;
};

std::map<int, Plan>& plans() {
  static std::map<int, Plan> p;
  return p;
}
std::map<std::string, Cfg>& tuned() {
  static std::map<std::string, Cfg> t;
  return t;
}

bool env_flag(const char* name, bool dflt) {
  const char* s = getenv(name);
  return s ? atoi(s) != 0 : dflt;
}

// a launcher enqueues the persistent kernel for config c on stream s; the
// kernels write the info of table entry p to info[p]
typedef void (*Launcher)(const Cfg& c, const void* ctx, const BDesc* tab, const void* extra, int nitems, int count,
                         unsigned* ctr, int* info, hipStream_t s);

void enqueue(Launcher L, const Cfg& c, const void* ctx, const BDesc* tab, const void* extra, int nitems, int count,
             unsigned* ctr, int* info, hipStream_t s) {
  bzero_kernel<<<1, BCTR, 0, s>>>(ctr, BCTR);
  L(c, ctx, tab, extra, nitems, count, ctr, info, s);
}

// Runs the batch `probs` through the cached graph of plan slot `slot`,
// re-capturing only when the table or config changed; `extra` makes the bytes
// that follow the table on the device and is only called then (the comparison
// and the work list took most of a call's 1 ms on the host at 10^4 problems).
// Returns the device info array.
template <typename Extra>
int* run_plan(int slot, Launcher L, const Cfg& c, const void* ctx, size_t ctx_bytes, const std::vector<BDesc>& probs,
              int nitems, const Extra& make_extra) {
  Runtime& r = rt();
  Plan& P = plans()[slot];
  const int count = (int)probs.size();
  const size_t tb = sizeof(BDesc) * probs.size();
  const bool use_graph = env_flag("OPENBLAS_AMD_BATCH_GRAPH", true);
  if (P.exec && use_graph && P.cfg.var == c.var && P.cfg.grid == c.grid && P.ctx.size() == ctx_bytes &&
      memcmp(P.ctx.data(), ctx, ctx_bytes) == 0 && P.probs.size() == probs.size() &&
      memcmp(P.probs.data(), probs.data(), tb) == 0) {
    OBA_HIP(hipGraphLaunch(P.exec, r.stream));
    return P.info.as<int>();
  }
  const std::vector<char> extra = make_extra();
  // the previous graph may still run from the last call: let it finish
  // before its table goes back to the pool
  OBA_HIP(hipStreamSynchronize(r.stream));
  if (P.exec) { OBA_HIP(hipGraphExecDestroy(P.exec)); P.exec = nullptr; }
  P.probs.clear();
  P.tab = DevBuf(tb + extra.size() + 16);
  P.ctr = DevBuf(sizeof(unsigned) * BCTR);
  P.info = DevBuf(sizeof(int) * (size_t)std::max(count, 1));
  OBA_HIP(hipMemcpyAsync(P.tab.p, probs.data(), tb, hipMemcpyHostToDevice, r.stream));
  if (!extra.empty())
    OBA_HIP(hipMemcpyAsync(P.tab.as<char>() + tb, extra.data(), extra.size(), hipMemcpyHostToDevice, r.stream));
  const BDesc* dt = P.tab.as<BDesc>();
  const void* dx = extra.empty() ? nullptr : (const void*)(P.tab.as<char>() + tb);
  if (!use_graph) {
    enqueue(L, c, ctx, dt, dx, nitems, count, P.ctr.as<unsigned>(), P.info.as<int>(), r.stream);
    return P.info.as<int>();
  }
  hipGraph_t g = nullptr;
  OBA_HIP(hipStreamBeginCapture(r.stream, hipStreamCaptureModeThreadLocal));
  enqueue(L, c, ctx, dt, dx, nitems, count, P.ctr.as<unsigned>(), P.info.as<int>(), r.stream);
  OBA_HIP(hipStreamEndCapture(r.stream, &g));
  OBA_HIP(hipGraphInstantiate(&P.exec, g, nullptr, nullptr, 0));
  OBA_HIP(hipGraphDestroy(g));
  P.cfg = c;
  P.ctx.assign((const char*)ctx, (const char*)ctx + ctx_bytes);
  P.probs = probs;
  OBA_HIP(hipGraphLaunch(P.exec, r.stream));
  return P.info.as<int>();
}

// Times every candidate config on scratch copies (operand a or b of each
// problem, rows x cols given by BDesc field indices) and keeps the fastest
// for this batch signature (Cholesky and solves).
Cfg tune(const std::string& sig, const std::vector<Cfg>& cands, Launcher L, const void* ctx,
         const std::vector<BDesc>& probs, bool b_operand, int rows_field, int cols_field, size_t elem) {
  auto& tt = tuned();
  auto f = tt.find(sig);
  if (f != tt.end()) return f->second;
  if (cands.size() == 1 || !env_flag("OPENBLAS_AMD_BATCH_TUNE", true)) { tt[sig] = cands[0]; return cands[0]; }
  Runtime& r = rt();
  const int count = (int)probs.size();
  // scratch copies of the in/out operand, packed
  std::vector<BDesc> scr = probs;
  size_t total = 0;
  for (auto& d : scr) {
    const int* fs = &d.m;
    total += elem * (size_t)std::max(fs[rows_field], 1) * (size_t)std::max(fs[cols_field], 1);
  }
  DevBuf sbuf(total + 256), tsrc(sizeof(BDesc) * count), tdst(sizeof(BDesc) * count),
      ctr(sizeof(unsigned) * BCTR), info(sizeof(int) * (size_t)std::max(count, 1));
  size_t off = 0;
  for (auto& d : scr) {
    const int* fs = &d.m;
    const int rows = std::max(fs[rows_field], 1);
    void* p = sbuf.as<char>() + off;
    off += elem * (size_t)rows * (size_t)std::max(fs[cols_field], 1);
    if (b_operand) { d.b = p; d.ldb = rows; }
    else { d.a = p; d.lda = rows; }
  }
  OBA_HIP(hipMemcpyAsync(tsrc.p, probs.data(), sizeof(BDesc) * count, hipMemcpyHostToDevice, r.stream));
  OBA_HIP(hipMemcpyAsync(tdst.p, scr.data(), sizeof(BDesc) * count, hipMemcpyHostToDevice, r.stream));
  auto refresh = [&]() {
    if (count == 0) return;
    dim3 g(64, (unsigned)count);
    if (elem == 8) bcopy_kernel<double><<<g, 256, 0, r.stream>>>(tsrc.as<BDesc>(), tdst.as<BDesc>(), b_operand, rows_field, cols_field);
    else bcopy_kernel<float><<<g, 256, 0, r.stream>>>(tsrc.as<BDesc>(), tdst.as<BDesc>(), b_operand, rows_field, cols_field);
  };
  hipEvent_t e0, e1;
  OBA_HIP(hipEventCreate(&e0));
  OBA_HIP(hipEventCreate(&e1));
  refresh();
  enqueue(L, cands[0], ctx, tdst.as<BDesc>(), nullptr, 0, count, ctr.as<unsigned>(), info.as<int>(), r.stream);
  float best = 1e30f;
  Cfg bc = cands[0];
  for (const Cfg& c : cands) {
    refresh();
    OBA_HIP(hipEventRecord(e0, r.stream));
    enqueue(L, c, ctx, tdst.as<BDesc>(), nullptr, 0, count, ctr.as<unsigned>(), info.as<int>(), r.stream);
    OBA_HIP(hipEventRecord(e1, r.stream));
    OBA_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    OBA_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (ms < best) { best = ms; bc = c; }
  }
  OBA_HIP(hipEventDestroy(e0));
  OBA_HIP(hipEventDestroy(e1));
  tt[sig] = bc;
  return bc;
}

std::string signature(int kind, size_t elem, int flags, const std::vector<BDesc>& probs) {
  long mx = 0, cnt = (long)probs.size();
  double work = 0;
  for (auto& d : probs) {
    mx = std::max<long>(mx, std::max(d.m, std::max(d.n, d.k)));
    work += (double)std::max(d.m, 1) * std::max(d.n, 1) * std::max(d.k, std::max(std::min(d.m, d.n), 1));
  }
  int lc = 0, lw = 0;
  while ((1L << lc) < cnt) lc++;
  while (work > 1.0 && lw < 80) { work /= 2; lw++; }
  char b[128];
  snprintf(b, sizeof b, "%d/%zu/%d/%d/%ld/%d", kind, elem, flags, lc, (mx + 31) / 32, lw);
  return b;
}

std::vector<char> no_extra() { return {}; }

int grid_of(const Cfg& c) { return std::max(1, rt().num_cu * c.grid); }

// ---- launchers ---------------------------------------------------------------
// nitems: the items of the longest segment
template <typename T, bool TA, bool TB>
void launch_gemm_form(const BDesc* tab, const void* extra, int nitems, unsigned* ctr, hipStream_t s) {
  static const int per_cu = [] {
    int n = 0;
    OBA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, bgemm_kernel<T, TA, TB>, 256, 0));
    return std::max(n, 1);
  }();
  const BSeg* seg = (const BSeg*)extra;
  bgemm_kernel<T, TA, TB><<<8 * std::min(nitems, std::max(rt().num_cu * per_cu / 8, 1)), 256, 0, s>>>(
      tab, seg, (const int2*)(seg + 1), ctr);
  OBA_HIP(hipGetLastError());
}

template <typename T>
void launch_gemm(const Cfg&, const void* ctx, const BDesc* tab, const void* extra, int nitems, int, unsigned* ctr,
                 int*, hipStream_t s) {
  const int ta = ((const int*)ctx)[0], tb = ((const int*)ctx)[1];
  if (!ta && !tb) launch_gemm_form<T, false, false>(tab, extra, nitems, ctr, s);
  else if (!ta && tb) launch_gemm_form<T, false, true>(tab, extra, nitems, ctr, s);
  else if (ta && !tb) launch_gemm_form<T, true, false>(tab, extra, nitems, ctr, s);
  else launch_gemm_form<T, true, true>(tab, extra, nitems, ctr, s);
}

// workgroups of a size class that the device holds at once
template <typename T, int NWV>
int getrf_slots() {
  static const int per_cu = [] {
    int n = 0;
    OBA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, bgetrf_kernel<T, NWV>, 64 * NWV, 0));
    return std::max(n, 1);
  }();
  return rt().num_cu * per_cu;
}

// one launch per size class: problems of up to 64, 128, 256 and 512 rows take
// as many threads as they have rows (classes joined by the caller: as the
// largest has)
template <typename T, int NWV>
void launch_getrf_class(const BDesc* tab, int first, int last, unsigned* ctr, int* info, hipStream_t s) {
  if (first == last) return;
  const int g = std::min(last - first, getrf_slots<T, NWV>());
  bgetrf_kernel<T, NWV><<<g, 64 * NWV, 0, s>>>(tab + first, last - first, ctr, info + first);
  OBA_HIP(hipGetLastError());
}

template <typename T>
void launch_getrf(const Cfg&, const void* ctx, const BDesc* tab, const void*, int, int count, unsigned* ctr,
                  int* info, hipStream_t s) {
  const int* end = (const int*)ctx;   // the classes' ends in the table, largest class first
  launch_getrf_class<T, 8>(tab, 0, end[0], ctr, info, s);
  launch_getrf_class<T, 4>(tab, end[0], end[1], ctr + 1, info, s);
  launch_getrf_class<T, 2>(tab, end[1], end[2], ctr + 2, info, s);
  launch_getrf_class<T, 1>(tab, end[2], count, ctr + 3, info, s);
}

template <typename T>
void launch_potrf(const Cfg& c, const void* ctx, const BDesc* tab, const void*, int, int count, unsigned* ctr,
                  int* info, hipStream_t s) {
  const int rpt = ((const int*)ctx)[0], lower = ((const int*)ctx)[1];
  const int g = grid_of(c);
#define OBA_BP(R, W, L) bpotrf_kernel<T, R, W, L><<<g, 256, 0, s>>>(tab, count, ctr, info)
  if (lower) {
    if (rpt == 1) { if (c.var == 0) OBA_BP(1, 16, true); else OBA_BP(1, 32, true); }
    else { if (c.var == 0) OBA_BP(2, 16, true); else OBA_BP(2, 32, true); }
  } else {
    if (rpt == 1) { if (c.var == 0) OBA_BP(1, 16, false); else OBA_BP(1, 32, false); }
    else { if (c.var == 0) OBA_BP(2, 16, false); else OBA_BP(2, 32, false); }
  }
#undef OBA_BP
  OBA_HIP(hipGetLastError());
}

template <typename T>
void launch_getrs(const Cfg& c, const void* ctx, const BDesc* tab, const void*, int, int count, unsigned* ctr, int*,
                  hipStream_t s) {
  const int S = ((const int*)ctx)[0], trans = ((const int*)ctx)[1];
  const int g = grid_of(c);
#define OBA_BS(SS)                                                                        \
  if (trans) bgetrs_kernel<T, SS, true><<<g, 256, 0, s>>>(tab, count, ctr);             \
  else bgetrs_kernel<T, SS, false><<<g, 256, 0, s>>>(tab, count, ctr);
  if (S == 1) { OBA_BS(1) } else if (S == 2) { OBA_BS(2) } else if (S == 4) { OBA_BS(4) } else { OBA_BS(8) }
#undef OBA_BS
  OBA_HIP(hipGetLastError());
}

template <typename T> constexpr int tslot(int kind) { return kind * 2 + (sizeof(T) == 8 ? 0 : 1); }

// dinfo[p] is the info of table entry p; the caller's slot is probs[p].idx
void collect_info(const int* dinfo, const std::vector<BDesc>& probs, int* info_host) {
  if (probs.empty()) return;
  Runtime& r = rt();
  std::vector<int> h(probs.size(), 0);
  OBA_HIP(hipMemcpyAsync(h.data(), dinfo, sizeof(int) * h.size(), hipMemcpyDeviceToHost, r.stream));
  OBA_HIP(hipStreamSynchronize(r.stream));
  for (size_t p = 0; p < probs.size(); p++) info_host[probs[p].idx] = h[p];
}

}  // namespace

// ---- drivers -------------------------------------------------------------------
template <typename T>
void gemm_batched(int ta, int tb, std::vector<BDesc>& probs) {
  if (probs.empty()) return;
  // work list: the tiles of every C, problem p's in segment p % 8
  BSeg seg{};
  int len[8] = {};
  for (size_t p = 0; p < probs.size(); p++) len[p & 7] += bgemm_tiles(probs[p].m) * bgemm_tiles(probs[p].n);
  for (int x = 0; x < 8; x++) seg.begin[x + 1] = seg.begin[x] + len[x];
  const int nw = seg.begin[8];
  auto work = [&]() {
    std::vector<char> wl(sizeof(BSeg) + sizeof(int2) * (size_t)nw);
    memcpy(wl.data(), &seg, sizeof seg);
    int2* at[8];
    for (int x = 0; x < 8; x++) at[x] = (int2*)(wl.data() + sizeof(BSeg)) + seg.begin[x];
    for (size_t p = 0; p < probs.size(); p++) {
      const int tiles = bgemm_tiles(probs[p].m) * bgemm_tiles(probs[p].n);
      for (int t = 0; t < tiles; t++) *at[p & 7]++ = make_int2((int)p, t);
    }
    return wl;
  };
  const int ctx[2] = {ta, tb};
  const Cfg c;
  double fl = 0, by = 0;
  for (auto& d : probs) {
    fl += 2.0 * d.m * d.n * d.k;
    by += sizeof(T) * ((double)d.m * d.k + (double)d.k * d.n + (d.beta != 0.0 ? 2.0 : 1.0) * d.m * d.n);
  }
  KTimer kt("batched_gemm", rt().stream, fl, by);
  run_plan(tslot<T>(BK_GEMM), launch_gemm<T>, c, ctx, sizeof ctx, probs, *std::max_element(len, len + 8), work);
}

template <typename T>
void getrf_batched(std::vector<BDesc>& probs, int* info_host) {
  // the kernel's size classes, largest first, each in the order given
  std::vector<unsigned char> cls(probs.size());
  int count[5] = {};
  double longest[4] = {}, sum[4] = {};   // of the problems' times (their unit cancels)
  for (size_t i = 0; i < probs.size(); i++) {
    const BDesc& d = probs[i];
    const int k = d.m > 512 ? 4 : d.m > 256 ? 0 : d.m > 128 ? 1 : d.m > 64 ? 2 : 3;
    cls[i] = (unsigned char)k;
    count[k]++;
    if (k == 4) continue;
    const double t = std::min(d.m, d.n) * (1.0 + 0.0025 * d.n);
    longest[k] = std::max(longest[k], t);
    sum[k] += t;
  }
  std::vector<BDesc> small(probs.size() - count[4]), big;
  int ctx[3], at[4] = {0};
  for (int k = 0; k < 3; k++) ctx[k] = at[k + 1] = at[k] + count[k];
  for (size_t i = 0; i < probs.size(); i++) {
    if (cls[i] < 4) small[at[cls[i]]++] = probs[i];
    else big.push_back(probs[i]);
  }
  // The launches run one after the other, which costs nothing where every class
  // fills the device.  A class joins the launch of the one above it where that
  // ends sooner by the time of the longest problem or of all of them over the
  // workgroups held at once (a problem alone: 36 us for 32 columns, 73 for 64,
  // 430 for 256, FP64).  A call with 600 problems of 8 to 200: 893 us in three
  // launches, 449 in one (846 with one queue of 256-thread workgroups, before the
  // classes); 10^4 of 8 to 256 keep three.
  {
    const double slots[4] = {(double)getrf_slots<T, 8>(), (double)getrf_slots<T, 4>(), (double)getrf_slots<T, 2>(),
                             (double)getrf_slots<T, 1>()};
    auto time = [&](int k, double more) { return std::max(longest[k], (sum[k] + more) / slots[k]); };
    for (int k = 0, c = 1; c < 4; c++) {
      if (sum[c] == 0) continue;
      if (sum[k] > 0 && time(k, sum[c]) < time(k, 0) + time(c, 0)) {
        sum[k] += sum[c];
        for (int e = k; e < std::min(c, 3); e++) ctx[e] = c < 3 ? ctx[c] : (int)small.size();
        if (c < 3) ctx[c] = ctx[k];
      } else {
        k = c;
      }
    }
  }
  if (!small.empty()) {
    const Cfg c;
    double fl = 0, by = 0;
    for (auto& d : small) {
      const double mm = d.m, nn = d.n, k = std::min(mm, nn);
      fl += mm * nn * k - (mm + nn) * k * k / 2.0 + k * k * k / 3.0;   // LU of m x n (LAPACK count, leading terms)
      by += 2.0 * sizeof(T) * mm * nn;
    }
    const int* di;
    {
      KTimer kt("batched_getrf", rt().stream, fl, by);
      di = run_plan(tslot<T>(BK_GETRF), launch_getrf<T>, c, ctx, sizeof ctx, small, 0, no_extra);
    }
    collect_info(di, small, info_host);
  }
  for (auto& d : big)
    info_host[d.idx] = getrf<T>(d.m, d.n, (T*)d.a, d.lda, d.ipiv, rt().stream);
}

template <typename T>
void potrf_batched(bool lower, std::vector<BDesc>& probs, int* info_host) {
  std::vector<BDesc> small, big;
  for (auto& d : probs) (d.n <= 512 ? small : big).push_back(d);
  if (!small.empty()) {
    int mx = 0;
    for (auto& d : small) mx = std::max(mx, d.n);
    const int ctx[2] = {mx <= 256 ? 1 : 2, lower ? 1 : 0};
    std::vector<Cfg> cands;
    for (int v = 0; v < 2; v++)
      for (int g : {1, 2, 4}) cands.push_back(Cfg{v, g});
    Cfg c = tune(signature(BK_POTRF, sizeof(T), ctx[0] * 2 + ctx[1], small), cands, launch_potrf<T>, ctx, small, false, 1,
                 1, sizeof(T));
    double fl = 0, by = 0;
    for (auto& d : small) {
      fl += (double)d.n * d.n * d.n / 3.0;
      by += sizeof(T) * (double)d.n * (d.n + 1);   // the triangle read and written
    }
    const int* di;
    {
      KTimer kt("batched_potrf", rt().stream, fl, by);
      di = run_plan(tslot<T>(BK_POTRF), launch_potrf<T>, c, ctx, sizeof ctx, small, 0, no_extra);
    }
    collect_info(di, small, info_host);
  }
  for (auto& d : big) info_host[d.idx] = potrf<T>(lower, d.n, (T*)d.a, d.lda, rt().stream);
}

template <typename T>
void getrs_batched(bool trans, std::vector<BDesc>& probs, int* info_host) {
  std::vector<BDesc> small, big;
  for (auto& d : probs) (d.n <= 512 ? small : big).push_back(d);
  for (auto& d : probs) info_host[d.idx] = 0;
  if (!small.empty()) {
    int mx = 0;
    for (auto& d : small) mx = std::max(mx, d.n);
    const int S = mx <= 64 ? 1 : mx <= 128 ? 2 : mx <= 256 ? 4 : 8;
    const int ctx[2] = {S, trans ? 1 : 0};
    std::vector<Cfg> cands;
    for (int g : {2, 4, 8, 16}) cands.push_back(Cfg{0, g});
    Cfg c = tune(signature(BK_GETRS, sizeof(T), ctx[0] * 2 + ctx[1], small), cands, launch_getrs<T>, ctx, small, true, 1,
                 2, sizeof(T));
    double fl = 0, by = 0;
    for (auto& d : small) {
      fl += 2.0 * d.n * d.n * std::max(d.k, 0);
      by += sizeof(T) * ((double)d.n * d.n + 2.0 * d.n * std::max(d.k, 0));
    }
    KTimer kt("batched_getrs", rt().stream, fl, by);
    run_plan(tslot<T>(BK_GETRS), launch_getrs<T>, c, ctx, sizeof ctx, small, 0, no_extra);
  }
  for (auto& d : big) {   // large problems: the single-problem solve
    Runtime& r = rt();
    std::vector<int> ipv((size_t)d.n), perm;
    OBA_HIP(hipMemcpyAsync(ipv.data(), d.ipiv, sizeof(int) * (size_t)d.n, hipMemcpyDeviceToHost, r.stream));
    OBA_HIP(hipStreamSynchronize(r.stream));
    ipiv_to_perm(d.n, ipv.data(), perm);
    DevBuf pb(sizeof(int) * perm.size());
    OBA_HIP(hipMemcpyAsync(pb.p, perm.data(), sizeof(int) * perm.size(), hipMemcpyHostToDevice, r.stream));
    getrs_perm<T>(trans, d.n, d.k, (const T*)d.a, d.lda, pb.as<int>(), (T*)d.b, d.ldb, r.stream);
    OBA_HIP(hipStreamSynchronize(r.stream));
  }
}

template void gemm_batched<double>(int, int, std::vector<BDesc>&);
template void gemm_batched<float>(int, int, std::vector<BDesc>&);
template void getrf_batched<double>(std::vector<BDesc>&, int*);
template void getrf_batched<float>(std::vector<BDesc>&, int*);
template void getrs_batched<double>(bool, std::vector<BDesc>&, int*);
template void getrs_batched<float>(bool, std::vector<BDesc>&, int*);
template void potrf_batched<double>(bool, std::vector<BDesc>&, int*);
template void potrf_batched<float>(bool, std::vector<BDesc>&, int*);

}  // namespace oba
