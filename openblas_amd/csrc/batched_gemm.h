// Batched GEMM kernel: one workgroup per tile of a C, the single GEMM's loads
// and main loop (gemm_tile.h).
//
// Work items (problem, tile of C) in 8 segments, one per XCD, largest problem
// first: a workgroup takes the items of its own XCD's segment (workgroup b runs
// on XCD b % 8), where the tiles of one problem meet its operands in that L2,
// then helps the others.  A segment's first items go to its workgroups as they
// are numbered, so a batch that fits the device has no queue; the counters lie
// on lines of their own and are only counted on where items are left (300
// products of 8 to 60: 50 us a call; 114 with every workgroup counting to the
// end of all eight counters on one line).  Tiles are 64 wide, 32 where no more than 32 rows
// (columns) are left or the problem has fewer than 64: a remainder pads to 32
// and, as every edge tile moves back inside its operand, most loads stay wide.
// Bound by the matrix cores (2*m*n*k plus the padding) and by the memory
// latency of short products: 10^4 square FP64 products of 8 to 256 took 3.62 ms
// with guarded loads of single elements and one queue, 2.48 ms now (35 TFLOP/s
// of the products themselves).  Three workgroups per CU (up to 22 VGPRs of the
// FP64 forms spill): a fourth spills more and takes 2.74 ms against 2.47, two
// leave the matrix cores waiting (2.70); 16-deep slabs for the 64x64 tile 2.60.
#pragma once
#include "gemm_tile.h"

namespace oba {

__host__ __device__ inline int bgemm_tiles(int n) { return n < 64 ? (n + 31) / 32 : (n + 63) / 64; }

template <typename T, int BM, int BN, bool TA, bool TB>
using BGemmTile = GemmTile<T, BM, BN, (BM == 64 && BN == 64 ? 64 : 128) / (int)sizeof(T), TA, TB>;

template <typename T, int BM, int BN, bool TA, bool TB>
__device__ __attribute__((always_inline)) inline void bgemm_tile(const BDesc& d, long mt, long nt, T* smem) {
  typedef BGemmTile<T, BM, BN, TA, TB> G;
  const long M = d.m, N = d.n, K = d.alpha != 0.0 ? d.k : 0;
  const long m0 = M >= BM ? min(mt, M - BM) : 0, n0 = N >= BN ? min(nt, N - BN) : 0;
  typename G::acc_t acc[G::FM][G::FN];
  G::product(acc, M, N, K, (const T*)(gptr<const T>)d.a, d.lda, (const T*)(gptr<const T>)d.b, d.ldb, m0, n0,
             (int)((K + G::BK_ - 1) / G::BK_), smem);
  G::store(acc, M, N, (T)d.alpha, (T)d.beta, (T*)(gptr<T>)d.c, d.ldc, mt, nt, m0, n0, 0);
}

struct BSeg {
  int begin[9];   // the segments' first items, then their end
  int pad[7];
};
constexpr int BG_CTR = 32;   // a segment's counter on a 128-byte line of its own

template <typename T, bool TA, bool TB>
__global__ __launch_bounds__(256, 3) void bgemm_kernel(const BDesc* __restrict__ desc, const BSeg* __restrict__ seg,
                                                       const int2* __restrict__ work, unsigned* __restrict__ counter) {
  __shared__ __attribute__((aligned(16))) T smem[BGemmTile<T, 64, 32, TA, TB>::STAGE];   // the largest
  __shared__ int s_item[2];
  // the grid's gridDim.x / 8 workgroups of a segment take its first items as
  // they are numbered; the counters count the items after those
  const int slots = gridDim.x >> 3;
  int sg = blockIdx.x & 7;   // thread 0: the segment it draws from
  auto next = [&]() {
    while (true) {
      const int i = seg->begin[sg] + slots + (int)atomicAdd(counter + BG_CTR * sg, 1u);
      if (i < seg->begin[sg + 1]) return i;
      // empty: one that is not, found by loads (every workgroup counting on to
      // the end of all eight took 60 us for 768 workgroups)
      unsigned c[8];
#pragma unroll
      for (int x = 0; x < 8; x++)
        c[x] = __hip_atomic_load(counter + BG_CTR * x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      int to = -1;
#pragma unroll
      for (int x = 0; x < 8; x++)
        if (to < 0 && seg->begin[x] + slots + (int)c[x] < seg->begin[x + 1]) to = x;
      if (to < 0) return -1;
      sg = to;
    }
  };
  bool more = false;   // a segment with more items than workgroups
#pragma unroll
  for (int x = 0; x < 8; x++) more = more || seg->begin[x + 1] - seg->begin[x] > slots;
  if (threadIdx.x == 0) {
    const int i = seg->begin[sg] + (int)(blockIdx.x >> 3);
    s_item[0] = i < seg->begin[sg + 1] ? i : more ? next() : -1;
  }
  __syncthreads();
  int cur = 0, it = s_item[0];
  while (it >= 0) {
    if (threadIdx.x == 0) s_item[cur ^ 1] = more ? next() : -1;   // read after the last barrier
    const int2 wk = work[it];
    const BDesc& d = desc[wk.x];
    const int tm = bgemm_tiles(d.m);
    const int mw = d.m < 64 ? 32 : 64, nw = d.n < 64 ? 32 : 64;
    const int mt = wk.y % tm * mw, nt = wk.y / tm * nw;
    const bool m32 = d.m - mt <= 32 || mw == 32, n32 = d.n - nt <= 32 || nw == 32;   // uniform
    if (!m32 && !n32) bgemm_tile<T, 64, 64, TA, TB>(d, mt, nt, smem);
    else if (!m32) bgemm_tile<T, 64, 32, TA, TB>(d, mt, nt, smem);
    else if (!n32) bgemm_tile<T, 32, 64, TA, TB>(d, mt, nt, smem);
    else bgemm_tile<T, 32, 32, TA, TB>(d, mt, nt, smem);
    __syncthreads();
    cur ^= 1;
    it = s_item[cur];
  }
}

}  // namespace oba
