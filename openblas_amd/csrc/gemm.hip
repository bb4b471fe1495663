// Level-3 GEMM for gfx950: C <- alpha*op(A)*op(B) + beta*C, column-major,
// FP64 on v_mfma_f64_16x16x4f64 and FP32 on v_mfma_f32_16x16x4f32.
//
// Reference semantics followed (not its blocking): the β pre-pass and the
// k==0 / α==0 early exit of driver/level3/level3.c:229-264, β==0 writing
// exact zeros (kernel/generic/gemm_beta.c:52), all four NN/NT/TN/TT forms of
// interface/gemm.c:87-111.
//
// Design (MI355X, not the GotoBLAS 5-loop): one workgroup of 4 wavefronts
// owns a BM x BN tile of C held in MFMA accumulators; K advances in BK slabs
// that are loaded from HBM with 16-byte vector loads into registers one slab
// ahead and staged through a double-buffered k-major LDS tile.  The MFMA is
// issued with op(B) as its first operand, and a lane's fragments are
// consecutive rows, so 16 lanes store 16 x 16 bytes of one column of C.  Tiles
// are mapped XCD-aware: the 8 XCDs each get a contiguous, grouped block of C
// tiles so that the panels of A and B they share stay in their own L2.
#include "kernels.h"
#include "gemm_tile.h"

namespace oba {

// the linear tile index of workgroup b: each of the 8 XCDs a contiguous range
__device__ inline int xcd_range(int b, int total) {
  const int x = b & 7, base = total >> 3, rem = total & 7;
  return x * base + min(x, rem) + (b >> 3);
}
// tile `lin` of the lower triangle of nt x nt tiles, in groups of 8 tile rows
// (columns left of a group's square first, down each column), so that equal
// ranges of lin are equal work: an order over the full square gave the last
// XCD twice the average share of the triangle (12000 x 448 FP64: 1810 us, and
// 1374 with the tiles dealt out one by one)
__device__ inline void tri_tile(int lin, int nt, int& tm, int& tn) {
  auto row_of = [](int i) {   // largest r with r(r+1)/2 <= i
    int r = (int)((sqrtf(8.0f * (float)i + 1.0f) - 1.0f) * 0.5f);
    while ((long)r * (r + 1) / 2 > i) r--;
    while ((long)(r + 1) * (r + 2) / 2 <= i) r++;
    return r;
  };
  const int g0 = row_of(lin) & ~7, gs = min(nt - g0, 8);
  const int off = lin - (int)((long)g0 * (g0 + 1) / 2);
  if (off < g0 * gs) {
    tm = g0 + off % gs;
    tn = off / gs;
  } else {
    const int o = off - g0 * gs, r = row_of(o);
    tm = g0 + r;
    tn = g0 + o - r * (r + 1) / 2;
  }
}

// KS > 1 (sliced K): the workgroup is KS groups of 4 wavefronts; group g
// multiplies the g-th of KS equal, BK-aligned k ranges into its own
// accumulators, and the KS partial tiles are summed in LDS in the fixed
// order 0..KS-1 before the epilogue (one launch, no workspace, the same
// result on every run).  It fills a CU with one workgroup when there are
// only about as many tiles as CUs.
template <typename T, int BM, int BN, int BK, bool TA, bool TB, int KS, int OCC>
__global__ __launch_bounds__(256 * KS, OCC) void gemm_kernel(long M, long N, long K, T alpha,
                                                      const T* __restrict__ A, long lda,
                                                      const T* __restrict__ B, long ldb, T beta,
                                                      T* __restrict__ C, long ldc, int tiles_m,
                                                      int tiles_n, int tri, const int* abort_flag,
                                                      long kc, long cstride) {
  // split K (gridDim.y parts, kc deep): part y multiplies its k range into
  // its own C buffer (cstride apart); a second kernel sums the parts
  if (kc > 0) {
    const long y = blockIdx.y;
    A += y * kc * (TA ? 1 : lda);
    B += y * kc * (TB ? ldb : 1);
    K = min(kc, K - y * kc);
    C += y * cstride;
  }
  typedef GemmTile<T, BM, BN, BK, TA, TB> G;
  typedef typename G::mf mf;
  typedef typename G::acc_t acc_t;
  constexpr int V = G::V, FM = G::FM, FN = G::FN, PM = G::PM, PN = G::PN;
  constexpr int STAGE = G::STAGE;   // one group's double-buffered slabs
  constexpr int SMEM = KS == 1 ? STAGE : (KS * STAGE > KS * BM * BN ? KS * STAGE : KS * BM * BN);
  __shared__ __attribute__((aligned(16))) T smem[SMEM];
  const int grp = KS == 1 ? 0 : (int)(threadIdx.x >> 8);
  T* const st = smem + grp * STAGE;
  long kg = 0;   // sliced K: the groups' common k-range length, a multiple of BK
  if (KS > 1) {
    kg = ((K + KS - 1) / KS + BK - 1) / BK * BK;
    A += grp * kg * (TA ? 1 : lda);
    B += grp * kg * (TB ? ldb : 1);
    K = max(0L, min(kg, K - grp * kg));
  }

  // XCD-aware tile order: workgroup b runs on XCD b%8; give each XCD a
  // contiguous range of the grouped tile order.
  int lin = xcd_range(blockIdx.x, gridDim.x);
  int tm, tn;
  if (tri) {   // gridDim.x = the tiles of the triangle
    tri_tile(lin, tiles_m, tm, tn);
    if (tri == 2) { const int x = tm; tm = tn; tn = x; }
  } else {
    constexpr int GM = 8;
    const int group = lin / (GM * tiles_n);
    const int first_m = group * GM;
    const int gsize = min(tiles_m - first_m, GM);
    const int in_group = lin - group * GM * tiles_n;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
  }
  // the tile owns C rows [mt, mt+BM) and columns [nt, nt+BN); an edge tile
  // reads from m0 = M-BM (n0 = N-BN) instead, where every load is in range,
  // recomputing rows of its neighbour that it does not store
  const long mt = (long)tm * BM, nt = (long)tn * BN;
  const long m0 = M >= BM ? min(mt, M - BM) : 0, n0 = N >= BN ? min(nt, N - BN) : 0;
  if (abort_flag && *abort_flag) return;

  const int lane = threadIdx.x & 63;
  const int wave = (threadIdx.x >> 6) & 3;
  const int wm0 = (wave & 1) * G::WTM, wn0 = (wave >> 1) * G::WTN;

  acc_t acc[FM][FN];
  const int nk = KS > 1 ? (int)(kg / BK) : (int)((K + BK - 1) / BK);
  G::product(acc, M, N, K, A, lda, B, ldb, m0, n0, nk, st);
  if constexpr (KS > 1) {
    const bool bz = (beta == T(0));
    // partial tiles to LDS (column-major BM x BN per group), then every
    // thread sums its elements over the groups in order and writes C
    __syncthreads();
    T* pt = smem + grp * BM * BN;
#pragma unroll
    for (int i = 0; i < FM; i += PM)
#pragma unroll
      for (int j = 0; j < FN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          typename AVec<T, PM>::type v;
#pragma unroll
          for (int e = 0; e < PM; e++) v[e] = acc[i + e][j][r];
          const int n = wn0 + (j / PN) * 16 * PN + PN * mf::orow(lane, r) + j % PN;
          *(typename AVec<T, PM>::type*)&pt[n * BM + wm0 + i * 16 + PM * (lane & 15)] = v;
        }
    __syncthreads();
    typedef typename AVec<T, V>::type vec;
#pragma unroll
    for (int e0 = threadIdx.x * V; e0 < BM * BN; e0 += 256 * KS * V) {
      const long m = m0 + e0 % BM, n = n0 + e0 / BM;
      vec sum = *(const vec*)&smem[e0];
#pragma unroll
      for (int g = 1; g < KS; g++) sum += *(const vec*)&smem[g * BM * BN + e0];
      if (n >= N || n < nt) continue;
      T* p = C + m + n * ldc;
#pragma unroll
      for (int e = 0; e < V; e++) {
        const long i = m + e;
        if (i < M && i >= mt && !(tri == 1 && n > i) && !(tri == 2 && i > n)) {
          T v = alpha * sum[e];
          if (!bz) v += beta * p[e];
          p[e] = v;
        }
      }
    }
  } else {
    G::store(acc, M, N, alpha, beta, C, ldc, mt, nt, m0, n0, tri);
  }
}

template <typename T>
__global__ void scale_kernel(long m, long n, T beta, T* c, long ldc) {
  long total = m * n;
  for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
    long i = idx % m, j = idx / m;
    T* p = c + i + j * ldc;
    *p = (beta == T(0)) ? T(0) : beta * *p;
  }
}

template <typename T>
void scale(long m, long n, T beta, T* c, long ldc, hipStream_t s) {
  if (m <= 0 || n <= 0 || beta == T(1)) return;
  long total = m * n;
  int blocks = (int)std::min<long>((total + 255) / 256, 4096);
  scale_kernel<T><<<blocks, 256, 0, s>>>(m, n, beta, c, ldc);
  OBA_HIP(hipGetLastError());
}

// C = alpha*A*B + beta*C with few columns (N <= GS_NMAX, no transposes):
// an HBM-bound matrix-vector product, where 64x64 MFMA tiles leave most of
// the device idle (one tile column: 1.36 ms for 16384^2 x 1 FP64, 6x the
// time to stream A).  Thread = row of A (coalesced down the columns), the k
// range cut into gridDim.y chunks for enough workgroups; the chunk's B
// values staged in LDS; per-chunk partial sums combined in chunk order by a
// second kernel (deterministic).
constexpr int GS_NMAX = 4;
constexpr int GS_KC = 256;   // B rows staged per LDS round

template <typename T, int NR>
__global__ __launch_bounds__(256) void gemm_skinny_part_kernel(long M, long K, long kchunk, const T* __restrict__ A,
                                                               long lda, const T* __restrict__ B, long ldb,
                                                               T* __restrict__ part) {
  __shared__ T sb[NR][GS_KC];
  const long i = blockIdx.x * 256L + threadIdx.x;
  const long k0 = (long)blockIdx.y * kchunk, k1 = min(K, k0 + kchunk);
  T acc[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) acc[r] = T(0);
  for (long kb = k0; kb < k1; kb += GS_KC) {
    const int kn = (int)min((long)GS_KC, k1 - kb);
    __syncthreads();
    for (int idx = threadIdx.x; idx < NR * GS_KC; idx += 256) {
      const int r = idx / GS_KC, kk = idx % GS_KC;
      sb[r][kk] = kk < kn ? B[kb + kk + r * ldb] : T(0);
    }
    __syncthreads();
    if (i < M) {
      const T* ap = A + i + kb * lda;
      int kk = 0;
      for (; kk + 8 <= kn; kk += 8) {   // 8 loads in flight
        T a[8];
#pragma unroll
        for (int u = 0; u < 8; u++) a[u] = ap[(long)(kk + u) * lda];
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
          for (int r = 0; r < NR; r++) acc[r] += a[u] * sb[r][kk + u];
      }
      for (; kk < kn; kk++) {
        const T a = ap[(long)kk * lda];
#pragma unroll
        for (int r = 0; r < NR; r++) acc[r] += a * sb[r][kk];
      }
    }
  }
  if (i < M) {
#pragma unroll
    for (int r = 0; r < NR; r++) part[((long)blockIdx.y * NR + r) * M + i] = acc[r];
  }
}

template <typename T, int NR>
__global__ __launch_bounds__(256) void gemm_skinny_sum_kernel(long M, int parts, const T* __restrict__ part, T alpha,
                                                              T beta, T* __restrict__ C, long ldc) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= M) return;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    T s = T(0);
    for (int p = 0; p < parts; p++) s += part[((long)p * NR + r) * M + i];
    T* cp = C + i + r * ldc;
    *cp = beta == T(0) ? alpha * s : alpha * s + beta * *cp;   // beta == 0: C is not read
  }
}

template <typename T, int NR>
static void gemm_skinny(long m, long k, T alpha, const T* a, long lda, const T* b, long ldb, T beta, T* c, long ldc,
                        hipStream_t s) {
  const long mb = (m + 255) / 256;
  const int parts = (int)std::max(1L, std::min((k + GS_KC - 1) / GS_KC, (4L * rt().num_cu + mb - 1) / mb));
  const long kchunk = ((k + parts - 1) / parts + GS_KC - 1) / GS_KC * GS_KC;
  const int np = (int)((k + kchunk - 1) / kchunk);
  DevBuf part(sizeof(T) * (size_t)np * NR * m);
  gemm_skinny_part_kernel<T, NR><<<dim3((unsigned)mb, (unsigned)np), 256, 0, s>>>(m, k, kchunk, a, lda, b, ldb,
                                                                                part.as<T>());
  OBA_HIP(hipGetLastError());
  gemm_skinny_sum_kernel<T, NR><<<(unsigned)mb, 256, 0, s>>>(m, np, part.as<T>(), alpha, beta, c, ldc);
  OBA_HIP(hipGetLastError());
}

template <typename T, int BM, int BN, int BK, int KS = 1, int OCC = 1>
static void launch_cfg(bool ta, bool tb, long M, long N, long K, T alpha, const T* A, long lda,
                       const T* B, long ldb, T beta, T* C, long ldc, hipStream_t s, int tri,
                       const int* abort_flag, int ksplit = 1, long kc = 0, long cstride = 0) {
  long tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  if (tm * tn > 0x7fffffffL) fatal("gemm: grid too large", nullptr);
  if (tri && (BM != BN || M != N)) fatal("gemm: a triangular update is of square tiles of a square C", nullptr);
  dim3 grid((unsigned)(tri ? tm * (tm + 1) / 2 : tm * tn), (unsigned)ksplit), block(256 * KS);
#define OBA_GEMM_L(TA_, TB_) \
  gemm_kernel<T, BM, BN, BK, TA_, TB_, KS, OCC><<<grid, block, 0, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, (int)tm, (int)tn, tri, abort_flag, kc, cstride)
  if (!ta && !tb) OBA_GEMM_L(false, false);
  else if (!ta && tb) OBA_GEMM_L(false, true);
  else if (ta && !tb) OBA_GEMM_L(true, false);
  else OBA_GEMM_L(true, true);
#undef OBA_GEMM_L
  OBA_HIP(hipGetLastError());
}

// C = sum of the ksplit partial products (alpha applied) + beta*C
template <typename T>
__global__ __launch_bounds__(256) void gemm_ksum_kernel(long M, long N, int parts, const T* __restrict__ W, T beta,
                                                        T* __restrict__ C, long ldc) {
  const long total = M * N;
  for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total; idx += (long)gridDim.x * 256) {
    T sum = T(0);
    for (int p = 0; p < parts; p++) sum += W[p * total + idx];
    const long i = idx % M, j = idx / M;
    T* cp = C + i + j * ldc;
    *cp = beta == T(0) ? sum : sum + beta * *cp;   // beta == 0: C is not read
  }
}

template <typename T>
void gemm(bool ta, bool tb, long m, long n, long k, T alpha, const T* a, long lda, const T* b,
          long ldb, T beta, T* c, long ldc, hipStream_t s, int tri, const int* abort_flag) {
  if (m <= 0 || n <= 0) return;
  if (k <= 0 || alpha == T(0)) {
    if (tri) fatal("gemm: triangular update with k==0 or alpha==0 is not supported", nullptr);
    scale<T>(m, n, beta, c, ldc, s);
    return;
  }
  // The split-K and few-column paths take a pool workspace.  Pool blocks are
  // ordered on the library stream only (a block freed there may be handed
  // out again before work queued on another stream has finished with it), so
  // a GEMM on any other stream (the look-ahead LU's trailing update) uses
  // the workspace-free tile kernels.
  const bool ws_ok = s == rt().stream;
  if (ws_ok && !ta && !tb && n <= GS_NMAX && tri == 0 && abort_flag == nullptr && m >= 2048 && k >= 2048) {
    switch (n) {
      case 1: gemm_skinny<T, 1>(m, k, alpha, a, lda, b, ldb, beta, c, ldc, s); return;
      case 2: gemm_skinny<T, 2>(m, k, alpha, a, lda, b, ldb, beta, c, ldc, s); return;
      case 3: gemm_skinny<T, 3>(m, k, alpha, a, lda, b, ldb, beta, c, ldc, s); return;
      default: gemm_skinny<T, 4>(m, k, alpha, a, lda, b, ldb, beta, c, ldc, s); return;
    }
  }
  // Tile, slab and K slicing by how many tiles there are per CU.  MI355X, us
  // per synchronous call (launch and completion about 10 us of it), NN unless
  // said; the last column is the kernel before this table (128x128 or 64x64
  // tiles, per-element loads at odd leading dimensions, fragments read in
  // front of their own MFMAs; 8192^3 on data that draw little power, normal
  // random data further down):
  //   FP64            64x64x8 KS1  KS2  64x32x16 KS2  32x32x16 KS1  KS2   before
  //   8192^3                15009  15300        16224         17668  18713  16400
  //   2047x3001x1501 TN       320    327          370           430    488    617
  //   4096x1024x4096          496    497          529           588    623    925
  //   2048x1024x2048          152    138          146           162    171    190
  //   256x5000x5000           346    303          258           263    258
  //   1024^3                   59     54           52            57     60     52
  //   512x1024x512             35     32           24            25     25     33
  //   512^3                    35     32           24            22     20     33
  //   64^3                   15.6   16.3         14.8          14.2   14.0   17.7
  // An FP64 MFMA takes 64 cycles, so a 64x64 tile hides its loads once a CU
  // holds several workgroups; with two tiles per CU or fewer a second wave
  // group per tile does that, and fewer tiles than CUs want smaller ones.
  constexpr bool D = sizeof(T) == 8;
  const long cu = rt().num_cu;
  const long m64 = (m + 63) / 64, m32 = (m + 31) / 32;   // tri: only the triangle's tiles run
  const long t64 = tri ? m64 * (m64 + 1) / 2 : m64 * ((n + 63) / 64), t6432 = m64 * ((n + 31) / 32);
  const long t32 = tri ? m32 * (m32 + 1) / 2 : m32 * ((n + 31) / 32);
  constexpr int BK32 = D ? 16 : 32, BK64 = D ? 8 : 16;
#define OBA_GEMM_ARGS ta, tb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s, tri, abort_flag
  if (8 * t64 < 7 * cu) {
    // A deep K of few tiles is split over workgroups too: 32x32 tiles with four
    // groups while two parts of them fit the CUs (256x256x8192 FP64: 95 us
    // unsplit, 33 in 16 parts), above that the tile and the parts that the
    // measured rates below make fastest: us per unit of k and tile (32x32 tiles
    // read both operands along k when op(A) is transposed and op(B) is not),
    // per round of two workgroups on a CU, for the sum and per byte of a part.
    // us per call, unsplit 32x32 / so split: FP64 640x256x4096 54 / 44,
    // 512x640x4096 83 / 65, 1280x400x2048 74 / 61, 640x1280x8192 308 / 231, FP32
    // 512x640x8192 114 / 64, 640x1280x1500 58 / 44; 512x1024x1024 stays at 32.
    // A C of at most 32 columns (rows) takes 64x32 (32x32) tiles, whose clamped
    // loads want two workgroups on a CU: 8192x28x4096 FP64 107 / 78, 16x5440x6528
    // FP32 92 / 63; below k = 2048 nothing is gained.
    if (ws_ok && tri == 0 && abort_flag == nullptr && k >= 1024) {
      const long parts_w = std::min<long>({8L, cu / std::max(t32, 1L), k / 512});
      long parts = 1, bm = 32, bn = 32;
      if (parts_w > 1) {
        parts = parts_w;
      } else if (std::min(m, n) <= 32) {
        if (n <= 32) bm = 64;
        double best = 1e300;
        for (long p = 1, t = n <= 32 ? t6432 : t32; p <= 12 && (p == 1 || (k >= 2048 && k >= 256 * p)); p++) {
          const double c = (double)((p * t + cu - 1) / cu), v = c / (double)p * (c == 1.0 ? 1.5 : 1.0);
          if (v < 0.97 * best) { best = v; parts = p; }
        }
      } else {
        const bool clamped = std::min(m, n) < 64;
        const double us64 = (D ? 0.033 : 0.0165) * (clamped ? 1.4 : 1.0);
        const double us32 = D ? (ta && !tb ? 0.0127 : 0.0095) : (ta && !tb ? 0.0071 : 0.0060);
        double best = 1e300;
        auto tile = [&](long w, long t, double us, double alone) {   // alone: the factor of one workgroup on its CU
          for (long p = 1; p <= 12 && (p == 1 || k >= 256 * p); p++) {
            const long c = (p * t + cu - 1) / cu;
            const double v = (double)(c * k) / (double)p * us * (c == 1 ? alone : 1.0) + 3.0 * (double)((c + 1) / 2) +
                             (p == 1 ? 0.0 : 4.5 + 3e-7 * (double)(p * m * n) * sizeof(T));
            if (v < best) { best = v; parts = p; bm = bn = w; }
          }
        };
        tile(32, t32, us32, D ? 1.1 : 1.0);   // unsplit: four groups
        tile(64, t64, us64, clamped ? 1.5 : 1.05);
      }
      if (parts > 1 || bm == 64) {
        if (parts > 1) {
          const long kc = ((k + parts - 1) / parts + 15) / 16 * 16;
          const int np = (int)((k + kc - 1) / kc);
          DevBuf w(sizeof(T) * (size_t)np * m * n);
#define OBA_GEMM_SPLIT ta, tb, m, n, k, alpha, a, lda, b, ldb, T(0), w.as<T>(), m, s, 0, nullptr, np, kc, m * n
          if (parts_w > 1) launch_cfg<T, 32, 32, BK32, 4, 2>(OBA_GEMM_SPLIT);
          else if (bm == 32) launch_cfg<T, 32, 32, BK32, 2, 2>(OBA_GEMM_SPLIT);
          else if (bn == 32) launch_cfg<T, 64, 32, BK32, 2, 2>(OBA_GEMM_SPLIT);
          else launch_cfg<T, 64, 64, BK64, 2, 2>(OBA_GEMM_SPLIT);
#undef OBA_GEMM_SPLIT
          const long total = m * n;
          gemm_ksum_kernel<T><<<(unsigned)std::min<long>((total + 255) / 256, 4096), 256, 0, s>>>(m, n, np, w.as<T>(), beta,
                                                                                                 c, ldc);
          OBA_HIP(hipGetLastError());
          return;
        }
        if (bn == 64) {
          launch_cfg<T, 64, 64, BK64, 2, 2>(OBA_GEMM_ARGS);
          return;
        }
      }
    }
    if (k >= 1024 && t32 <= cu) launch_cfg<T, 32, 32, BK32, 4, 2>(OBA_GEMM_ARGS);
    else if (k >= 1024 || (k >= (D ? 256 : 512) && t32 <= 2 * cu)) launch_cfg<T, 32, 32, BK32, 2, 2>(OBA_GEMM_ARGS);
    else launch_cfg<T, 32, 32, BK32, 1, 4>(OBA_GEMM_ARGS);
    return;
  }
  if (D && tri == 0 && t64 <= 4 * cu && k >= 256) {
    // the narrower tile where 64x64 ones would fill their last round of CUs
    // worse (316 tiles on 256 CUs: 303 us, 632 half tiles: 258), or there is
    // one per CU
    auto fill = [cu](long t) { return (double)t / (double)((t + cu - 1) / cu * cu); };
    if (t64 <= cu || 0.95 * fill(t6432) > fill(t64)) {
      if (t64 <= 2 * cu) launch_cfg<T, 64, 32, BK32, 2, 2>(OBA_GEMM_ARGS);
      else launch_cfg<T, 64, 32, BK32, 1, 4>(OBA_GEMM_ARGS);
      return;
    }
  }
  // FP32 (16-cycle steps) needs the LDS reuse of 128x128 tiles once there are
  // enough of them: 8192^3 7883 us against 8414 with 64x64; 3000^3 574 / 468.
  // With fewer they pay where their rounds of two per CU come out full (128x128
  // / 64x64, us): NN 4096^3 1018 / 1069, 4096x2048x1000 141 / 149, TT 4096^3 1006
  // / 1155, 8192x2048x200 74 / 78, 5440x4096x1000 (0.90 full) 390 / 403; not NN
  // 5440x4096x1000 392 / 376, 5000^3 (0.78) 2140 / 2051, TT 3500^3 (0.77) 865 / 753.
  // Nor below k = 128, where the tail's clamped loads show: 8192x5440x24 65 / 56.
  // FP64 gains from them at the largest sizes only, where 64x64 tiles read A and
  // B 40 times over (normal random data, 64x64x8 / 128x128x8 / 128x128x4, ms):
  // 8192^3 16.43 (17.7 on a card whose memory is slower) / 15.63 / 15.82, 6000^3
  // 6.78 / 6.56 / 6.58, 4000^3 1.97 / 1.98 / 1.94, 6144^2 x 2048 2.25 / 2.28 /
  // 2.30, 12000^2 x 448 2.00 / 2.20 / 2.12.  The FP64 form spills 194 to 256
  // VGPRs around its tail and its stores; the main loop reads none of them back.
  const long m128 = (m + 127) / 128, t128 = tri ? m128 * (m128 + 1) / 2 : m128 * ((n + 127) / 128);
  const long slots = 2 * cu, rounds = (t128 + slots - 1) / slots;
  const bool full128 = !D && tri == 0 && k >= 128 && t128 >= slots && t128 >= (ta && tb ? 0.85 : 0.95) * (double)(rounds * slots);
  if (t64 <= 2 * cu && k >= 256) launch_cfg<T, 64, 64, BK64, 2, 2>(OBA_GEMM_ARGS);
  else if (full128 || (t128 >= 8 * cu && (D ? tri == 0 && k >= 4096 : k >= 128))) launch_cfg<T, 128, 128, D ? 8 : 16, 1, 2>(OBA_GEMM_ARGS);
  else launch_cfg<T, 64, 64, BK64, 1, 4>(OBA_GEMM_ARGS);
#undef OBA_GEMM_ARGS
}

template void gemm<double>(bool, bool, long, long, long, double, const double*, long, const double*, long, double, double*, long, hipStream_t, int, const int*);
template void gemm<float>(bool, bool, long, long, long, float, const float*, long, const float*, long, float, float*, long, hipStream_t, int, const int*);
template void scale<double>(long, long, double, double*, long, hipStream_t);
template void scale<float>(long, long, float, float*, long, hipStream_t);

}  // namespace oba
