// Batched LU kernel: one workgroup of NWV wavefronts factors one problem of up
// to 64*NWV rows (partial pivoting, the rules of lapack/getf2/getf2_k.c) in
// 32-column panels, problems taken from an atomic queue.
//
// Per panel:
//  * thread t holds row j0+t of the panel in registers.  A column costs two
//    barriers: the wavefronts' best keys, then the pivot row, which its own
//    lane lays into LDS.  The update reads that row once, an element per lane,
//    and broadcasts it inside the FMA (DPP), so an element costs one
//    instruction and no LDS read.  Multipliers go straight to memory at the
//    row they have; the columns run in blocks of 8 with fixed registers, rows
//    shifting by 8 registers after a block.
//  * the rows that moved are put right at once (rows stay in LAPACK order, so
//    later panels and tiles shrink with the matrix): one load instruction per
//    column gathers the pivots' rows (lanes 0..31) and the rows they displace
//    (lanes 32..63, stored to their new places), in the panel and right of it;
//    U12 is a substitution with one column per thread; A22 -= L21 U12 runs on
//    MFMA 16x16 tiles, the next tile's elements in flight;
//  * the columns left of the panel are permuted once, at the end.
// Bound by the column chain's latency: 10^4 FP64 problems of 8 to 256 rows
// took 13.75 ms with a row permutation kept in LDS, panels of 8 or 16 columns
// and 256 threads whatever the rows, 4.6 ms now; of a problem's time the
// columns are 39 % (about 2300 cycles each with 3 workgroups on a CU, 1900
// alone), the trailing update 25 %, the gathers 13 %.  16-column panels take
// 5.8 ms instead of 3.9 for the problems above 128 rows (twice the passes over
// the trailing matrix), a fourth workgroup per CU 4.0 (the FP64 forms of 4 and 8
// wavefronts spill 5 VGPRs with three, more with four).
#pragma once
#include "lu_key.h"
#include "wave.h"

namespace oba {

constexpr int BLU_W = 32;

// x[0..N-1] += (u of lanes L0.. of each 16-lane row) * l, the broadcast taken
// by the FMA itself (DPP row_newbcast): no LDS read and no move per element.
// The leading s_nop covers the two wait states between a VALU write of u and
// its DPP read, which the compiler does not see inside the block.
#define BLU_DPP(T, D, U, L, K) "v_fmac_" T "_dpp %" #D ", %" #U ", %" #L " row_newbcast:%" #K " row_mask:0xf bank_mask:0xf\n\t"
template <int L0, int N>
__device__ __attribute__((always_inline)) inline void blu_fmac(double* x, double u, double l) {
  if constexpr (N >= 4) {
    asm("s_nop 1\n\t" BLU_DPP("f64", 0, 4, 5, 6) BLU_DPP("f64", 1, 4, 5, 7) BLU_DPP("f64", 2, 4, 5, 8) BLU_DPP("f64", 3, 4, 5, 9)
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3])
        : "v"(u), "v"(l), "n"(L0), "n"(L0 + 1), "n"(L0 + 2), "n"(L0 + 3));
    blu_fmac<L0 + 4, N - 4>(x + 4, u, l);
  } else if constexpr (N >= 1) {
    asm("s_nop 1\n\t" BLU_DPP("f64", 0, 1, 2, 3) : "+v"(x[0]) : "v"(u), "v"(l), "n"(L0));
    blu_fmac<L0 + 1, N - 1>(x + 1, u, l);
  }
}
template <int L0, int N>
__device__ __attribute__((always_inline)) inline void blu_fmac(float* x, float u, float l) {
  if constexpr (N >= 4) {
    asm("s_nop 1\n\t" BLU_DPP("f32", 0, 4, 5, 6) BLU_DPP("f32", 1, 4, 5, 7) BLU_DPP("f32", 2, 4, 5, 8) BLU_DPP("f32", 3, 4, 5, 9)
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3])
        : "v"(u), "v"(l), "n"(L0), "n"(L0 + 1), "n"(L0 + 2), "n"(L0 + 3));
    blu_fmac<L0 + 4, N - 4>(x + 4, u, l);
  } else if constexpr (N >= 1) {
    asm("s_nop 1\n\t" BLU_DPP("f32", 0, 1, 2, 3) : "+v"(x[0]) : "v"(u), "v"(l), "n"(L0));
    blu_fmac<L0 + 1, N - 1>(x + 1, u, l);
  }
}
#undef BLU_DPP

// U12 of one column in registers: u[i] -= L11(i, K) u[K] for i > K; the
// strictly lower L11 in LDS, column K across the lanes of each 16-lane row
template <int K, typename T, int LDD>
__device__ __attribute__((always_inline)) inline void blu_solve(T* u, const T* l11, int lr) {
  if constexpr (K < BLU_W - 1) {
    if constexpr (K < 15) blu_fmac<K + 1, 15 - K>(u + K + 1, l11[lr * LDD + K], -u[K]);
    constexpr int I0 = K < 15 ? 16 : K + 1;
    blu_fmac<I0 - 16, BLU_W - I0>(u + I0, l11[(16 + lr) * LDD + K], -u[K]);
    blu_solve<K + 1, T, LDD>(u, l11, lr);
  }
}

// the state of a thread's panel row and of its workgroup's column loop
template <typename T> struct BLuPanel {
  T x[BLU_W];          // column jb + c of the row, jb the current block of 8 columns
  int pos;             // the row's position from the panel's first row, -1: no row
  int morig, mcur;     // wavefront 0: see the kernel
  int info;
};

// column jb + JJ of a panel
template <int JJ, typename T, int NWV, int LDU>
__device__ __attribute__((always_inline)) inline void blu_column(BLuPanel<T>& p, int jb, int j0, int w0, bool act, int w,
                                                                 T* s_u, LuCand<T>* s_k, T* s_rv, gptr<T>& mul,
                                                                 gptr<int> ipiv) {
  constexpr int W = BLU_W;
  typedef typename LuKey<T>::U KU;
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, j = jb + JJ;
  KU key = 0;
  unsigned npos = 0;
  int win = 0;
  if (act) {
    const bool live = p.pos >= j;
    key = live ? LuKey<T>::key(p.x[JJ], p.pos == j) : KU(0);
    npos = live ? ~(unsigned)p.pos : 0u;
    win = l3_best_lane(key, npos);
  }
  if (lane == win) {
    LuCand<T> cd;
    cd.key = key;
    cd.npos = npos;
    s_k[w] = cd;
  }
  __syncthreads();
  LuCand<T> best = s_k[0];
  int bw = 0;
#pragma unroll
  for (int v = 1; v < NWV; v++) {
    const LuCand<T> cc = s_k[v];
    const bool tk = cc.beats(best);
    best.key = tk ? cc.key : best.key;
    best.npos = tk ? cc.npos : best.npos;
    bw = tk ? v : bw;
  }
  const int gp = (int)__builtin_amdgcn_readfirstlane(~best.npos);
  T* const urow = s_u + j * LDU;
  if (w == __builtin_amdgcn_readfirstlane(bw) && lane == win) {
#pragma unroll
    for (int c = JJ; c < 16; c++) urow[c] = p.x[c];
    if (w0 - jb > 16) {
#pragma unroll
      for (int c = 16; c < W; c++) urow[c] = p.x[c];
    }
    const T a = p.x[JJ];
    s_rv[0] = (a != T(0) && fabs(a) >= MinNormal<T>::v) ? T(1) / a : T(1);
  }
  __syncthreads();
  if (w == 0) {
    const bool fresh = gp >= w0 && __ballot(p.morig == gp) == 0;
    if (fresh && lane == W + j) p.morig = p.mcur = gp;
    p.mcur = p.mcur == gp ? j : (p.mcur == j ? gp : p.mcur);
    if (lane == 0) ipiv[j0 + j] = j0 + gp + 1;
    if (p.info == 0 && best.key == KU(1)) p.info = j0 + j + 1;   // key 1: zero
  }
  if (act) {
    const T ua = urow[lr], ub = urow[16 + lr];
    p.pos = p.pos == gp ? j : (p.pos == j ? gp : p.pos);
    const T l = p.x[JJ] * s_rv[0];
    if (p.pos > j) mul[(unsigned)t] = l;   // at the row it had; rows that moved are put right after the panel
    blu_fmac<JJ + 1, 15 - JJ>(p.x + JJ + 1, ua, -l);
    if (w0 - jb > 16) blu_fmac<0, 16>(p.x + 16, ub, -l);
  }
}

template <int JJ, typename T, int NWV, int LDU, typename M>
__device__ __attribute__((always_inline)) inline void blu_columns(BLuPanel<T>& p, int jb, int j0, int w0, bool act, int w,
                                                                  T* s_u, LuCand<T>* s_k, T* s_rv, M& mul, long lda,
                                                                  gptr<int> ipiv) {
  if constexpr (JJ < 8) {
    if (jb + JJ < w0) {
      blu_column<JJ, T, NWV, LDU>(p, jb, j0, w0, act, w, s_u, s_k, s_rv, mul, ipiv);
      mul += lda;
      blu_columns<JJ + 1, T, NWV, LDU>(p, jb, j0, w0, act, w, s_u, s_k, s_rv, mul, lda, ipiv);
    }
  }
}

template <typename T, int NWV>
__global__ __launch_bounds__(64 * NWV, NWV <= 2 ? 2 : 3) void bgetrf_kernel(const BDesc* __restrict__ desc, int count,
                                                             unsigned* __restrict__ counter,
                                                             int* __restrict__ info_out) {
  constexpr int W = BLU_W, NT = 64 * NWV, LDU = W + 4, CC = NWV < 4 ? 32 * NWV : 128, LDC = CC + 1;
  constexpr int LDD = W + 1, MAXP = NT / W, G = 8;
  typedef MF<T> mf;
  __shared__ T s_c[W * LDC];                // U12 of a column chunk
  __shared__ T s_l[W * LDD];                // strictly lower part of the diagonal block
  __shared__ __attribute__((aligned(16))) T s_u[W * LDU];   // pivot row j, element c: column (j & ~7) + c of the panel
  __shared__ __attribute__((aligned(16))) LuCand<T> s_k[NWV];
  __shared__ T s_rv[1];
  __shared__ short s_src[MAXP][2 * W];      // per panel, from its first row: lane i < W: the row that came to
  __shared__ short s_dst[MAXP][2 * W];      // position i; lanes from W: displaced rows and where they went (-1: none)
  __shared__ short s_map[NT];
  __shared__ int s_next;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), lr = lane & 15, lg = lane >> 4;

  if (t == 0) s_next = (int)atomicAdd(counter, 1u);
  __syncthreads();
  int it = s_next;
  while (it < count) {
    const BDesc& d = desc[it];
    const int m = d.m, n = d.n, kmax = min(d.m, d.n);
    const long lda = d.lda;
    gptr<T> A = (gptr<T>)d.a;
    gptr<int> ipiv = (gptr<int>)d.ipiv;
    int np = 0;
    BLuPanel<T> p;
    p.info = 0;
    __syncthreads();
    if (t == 0) s_next = (int)atomicAdd(counter, 1u);   // the next problem, read after the last barrier
#pragma unroll 1
    for (int j0 = 0; j0 < kmax; j0 += W, np++) {
      const int w0 = min(W, kmax - j0), mp = m - j0;
      const bool act = 64 * w < mp;   // this wavefront has rows
      p.pos = t < mp ? t : -1;
      gptr<T> P = A + j0 + (long)j0 * lda;   // the panel
      if (act) {
        gptr<const T> src = (gptr<const T>)P;
        const unsigned tr = (unsigned)min(t, mp - 1);
#pragma unroll
        for (int c = 0; c < W; c++) {
          p.x[c] = src[tr];
          src += c < w0 - 1 ? lda : 0;
        }
      } else {
#pragma unroll
        for (int c = 0; c < W; c++) p.x[c] = T(0);
      }
      // lane i < w0 of wavefront 0 follows the row that was at position i, lane
      // W+j the one first found at the pivot position of column j when that is
      // >= w0
      p.morig = p.mcur = lane < w0 ? lane : -1;
#pragma unroll
      for (int c = 0; c < W; c++) asm volatile("" : "+v"(p.x[c]));   // the loads are awaited here, not in the loop
      gptr<T> mul = P;
#pragma unroll 1
      for (int jb = 0; jb < w0; jb += 8) {
        blu_columns<0, T, NWV, LDU>(p, jb, j0, w0, act, w, s_u, s_k, s_rv, mul, lda, ipiv);
#pragma unroll
        for (int c = 0; c < W; c++) p.x[c] = c + 8 < W ? p.x[c + 8] : T(0);
      }
      const int morig = p.morig, mcur = p.mcur;
      if (w == 0) {
        // displaced rows end at positions >= w0 and come from the first w0
        const bool mv = lane < W && mcur >= w0;
        const unsigned long long mm = __ballot(mv);
        if (morig >= 0 && mcur < w0) s_src[np][mcur] = (short)morig;
        if (lane < 2 * W) s_dst[np][lane] = lane < w0 ? (short)lane : (short)-1;
        if (mv) {
          const int k = W + __popcll(mm & ((1ull << lane) - 1));
          s_src[np][k] = (short)morig;
          s_dst[np][k] = (short)mcur;
        }
      }
      __syncthreads();
      const int dst = lane < 2 * W ? s_dst[np][lane] : -1;
      const unsigned src = dst >= 0 ? (unsigned)s_src[np][lane] : 0u;
      // the panel's own columns: the pivots' rows (multipliers, then the rows
      // of U) and the multipliers of the rows they displaced
#pragma unroll 1
      for (int c = w; c < w0; c += G * NWV) {
        T v[G];
#pragma unroll
        for (int u = 0; u < G; u++) v[u] = (P + (long)min(c + u * NWV, w0 - 1) * lda)[src];
#pragma unroll
        for (int u = 0; u < G; u++) {
          const int cu = c + u * NWV;
          if (cu < w0) {
            if (lane < W) {
              s_l[lane * LDD + cu] = cu < lane ? v[u] : T(0);
              if (cu >= lane) v[u] = s_u[lane * LDU + cu - (lane & ~7)];
            }
            if (dst >= 0) (P + (long)cu * lda)[(unsigned)dst] = v[u];
          }
        }
      }
      __syncthreads();
      const int c1 = j0 + w0, nr = m - c1, nc = n - c1;
#pragma unroll 1
      for (int cb = 0; cb < nc; cb += CC) {
        const int cw = min(CC, nc - cb);
        gptr<T> C = A + (long)(c1 + cb) * lda + j0;
        // the pivots' rows to LDS, the rows they displace to their places
#pragma unroll 1
        for (int c = w; c < cw; c += G * NWV) {
          T v[G];
#pragma unroll
          for (int u = 0; u < G; u++) v[u] = (C + (long)min(c + u * NWV, cw - 1) * lda)[src];
#pragma unroll
          for (int u = 0; u < G; u++) {
            const int cu = c + u * NWV;
            if (cu < cw) {
              if (lane < W) s_c[lane * LDC + cu] = lane < w0 ? v[u] : T(0);
              else if (dst >= 0) (C + (long)cu * lda)[(unsigned)dst] = v[u];
            }
          }
        }
        __syncthreads();
        if (64 * w < cw) {   // U12, one column per thread; every lane takes part in the broadcasts
          const int tc = min(t, cw - 1);
          T u[W];
#pragma unroll
          for (int k = 0; k < W; k++) u[k] = s_c[k * LDC + tc];
          blu_solve<0, T, LDD>(u, s_l, lr);
          if (t < cw) {
#pragma unroll
            for (int k = 0; k < W; k++) s_c[k * LDC + t] = u[k];
          }
        }
        __syncthreads();
        for (int i = t; i < W * cw; i += NT) {
          const int r = i % W, c = i / W;
          if (r < w0) C[r + (long)c * lda] = s_c[r * LDC + c];
        }
        // A22 -= L21 U12, a 16-row tile after the other; the multipliers come
        // back from memory (cache) as fragments
#pragma unroll 1
        for (int r0 = 16 * w; r0 < nr; r0 += 16 * NWV) {
          const int rr = r0 + lr;
          const bool in = rr < nr;
          T fa[W / 4];
          {
            gptr<const T> l = (gptr<const T>)P + w0 + min(rr, nr - 1) + (long)lg * lda;
#pragma unroll
            for (int k = 0; k < W / 4; k++) {
              fa[k] = -*l;
              l += 4 * lda;
            }
          }
          gptr<T> q = C + w0 + min(rr, nr - 1);
          typename mf::acc acc, nxt;
          auto load = [&](int ct, typename mf::acc& v) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = q[(long)min(ct + mf::orow(lane, e), cw - 1) * lda];
          };
          load(0, acc);
#pragma unroll 1
          for (int ct = 0; ct < cw; ct += 16) {
            load(min(ct + 16, cw - 1), nxt);
            T fb[W / 4];
#pragma unroll
            for (int k = 0; k < W / 4; k++) fb[k] = s_c[(4 * k + lg) * LDC + min(ct + lr, cw - 1)];
#pragma unroll
            for (int k = 0; k < W / 4; k++) acc = mf::mma(fb[k], fa[k], acc);
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (in && ct + mf::orow(lane, e) < cw) q[(long)(ct + mf::orow(lane, e)) * lda] = acc[e];
            acc = nxt;
          }
        }
        __syncthreads();
      }
    }
    // the columns left of each panel: the later panels' interchanges, from the
    // last one back (thread i: row i comes from row `from`)
    int from = t;
#pragma unroll 1
    for (int b = np - 1; b > 0; b--) {
      const int jb = b * W;
      s_map[t] = (short)t;
      __syncthreads();
      if (t < 2 * W) {
        const int dd = s_dst[b][t];
        if (dd >= 0) s_map[jb + dd] = (short)(jb + s_src[b][t]);
      }
      __syncthreads();
      from = s_map[from];
      const bool mv = t < m && from != t;
#pragma unroll 1
      for (int c0 = jb - W; c0 < jb; c0 += G) {
        gptr<T> L = A + (long)c0 * lda;
        T v[G];
        if (mv) {
#pragma unroll
          for (int c = 0; c < G; c++) v[c] = (L + c * lda)[(unsigned)from];
        }
        __syncthreads();
        if (mv) {
#pragma unroll
          for (int c = 0; c < G; c++) (L + c * lda)[(unsigned)t] = v[c];
        }
      }
    }
    if (t == 0) info_out[it] = p.info;
    __syncthreads();
    it = s_next;
  }
}

}  // namespace oba
