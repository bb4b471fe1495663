// The LU leaf panel kernel for panels of up to L3_PMAX workgroups (16384
// rows): factors A(j0:m, j0:j0+w) held as At(j0:j0+w, j0:m), w <= 32, with
// partial pivoting (IAMAX order and NaN rule of kernel/arm/iamax.c:51-74).
//
// A column is a chain of dependent steps (find the pivot over all rows, hand
// its row to every workgroup, update), so the kernel is bound by the latency
// of that chain, not by flops or bytes.  Measured per 32-column launch,
// MI355X, against lu_panel_kernel: FP32 512 rows 87.8 -> 45.7 us, 4096 rows
// 131 -> 83, 16384 rows 152 -> 90; FP64 88.7 -> 56.7, 147 -> 94, 167 -> 109.
// What the chain consists of, in cycles of 2.4 GHz (FP32, 16384 rows): the
// wavefront's best key 365, workgroup's best 260, its row to memory 260, the
// records' travel 2500, best of a wavefront's records 550, of all 850 (with
// the wait for the slowest wavefront), multipliers and next column 250.
//  * 256 threads (one wavefront per SIMD) with two rows each: every fixed
//    per-wavefront cost (reductions, broadcasts, barriers) is paid by 4
//    wavefronts instead of 8.
//  * A row is y[k] = column j+k: the update of column j writes element k+1
//    into register k, so the column loop is one compact body with static
//    register indices and no moves; finished multipliers go to LDS, finished
//    rows of U too, and rows are put together when they are written back.
//  * The update by column j-1 of everything but the next column runs after
//    column j's candidate has left, behind the exchange; the published row
//    gets the same update (same operands, one rounding) on its way out.
//  * Only the key and position of a wavefront's best row go through the first
//    barrier; the winning wavefront alone lays its row out over the lanes.
//  * A record is plain data, no tags: its words start as L3_EMPTY and are
//    written once, each 8-byte store seen whole or not at all, so a record is
//    complete when no word is L3_EMPTY.  Tagged words were twice the bytes,
//    and the travel time grows with the lines moved (a header line of its own
//    per record cost +2500 cycles a column).  Each column has its own
//    records; a panel's kernel empties those of the next.
//  * 1/pivot is taken by every lane for its own candidate beside the
//    wavefront reduction and travels with the record: the division is off the
//    chain.
//  * The records of the workgroups spread over all XCDs: keeping the panel on
//    one XCD was measured no faster (P = 16: 104 against 100 us).
#pragma once

constexpr int L3_NT = 256, L3_NW = 4, L3_RPT = 2, L3_ROWS = L3_NT * L3_RPT;
constexpr int L3_PMAX = 32;   // workgroups; a wavefront polls up to L3_PMAX / L3_NW records at once
constexpr unsigned long long L3_EMPTY = ~0ull;

// one candidate record: header words, then the row from the current column on
template <typename T> struct L3Rec {
  static constexpr int HW = sizeof(T) / 4;               // FP32 {rinv, npos}; FP64 {0, npos}, rinv
  static constexpr int RW = LU_W * (int)sizeof(T) / 8;   // row words
  static constexpr int N = sizeof(T) == 8 ? 40 : 24;     // stride: whole 64-byte lines
  static constexpr size_t COL = (size_t)L3_PMAX * N;     // words of a column's records
  static constexpr size_t AREA = LU_W * COL;             // of a panel's (two areas, used in turn)
};

template <typename T, int W, bool MULTI>
__global__ __launch_bounds__(L3_NT) void lu_panel3_kernel(T* __restrict__ At, long ldt, long m, long j0, int w,
                                                          int* __restrict__ ipiv, int* __restrict__ info,
                                                          int* __restrict__ moves, unsigned long long* __restrict__ rec,
                                                          unsigned long long* __restrict__ rec_next, unsigned* err,
                                                          int pre) {
  typedef typename LuKey<T>::U KU;
  typedef LuCand<T> Cand;
  typedef L3Rec<T> R;
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
  constexpr int V = 16 / sizeof(T);
  constexpr int NW = L3_NW, RPT = L3_RPT, ROWS = L3_ROWS, WR = ROWS / NW;
  constexpr int LDL = ROWS + 1, LDU = W + 4, LDU12 = W + 1;
  constexpr int RPI = 64 / R::RW;              // records per load instruction
  constexpr int NR = L3_PMAX / NW;             // records per wavefront
  constexpr int NL = NR / RPI;
  constexpr unsigned FAIL = 1u;                // npos of a wait that ran out (no position has it)
  static_assert(W == LU_W && W == 32, "");
  __shared__ T s_l[W * LDL];                   // multipliers, element (c, row) at c*LDL + row
  __shared__ __attribute__((aligned(16))) T s_u[(W + 1) * LDU];        // pivot row j, from its diagonal on, in row j+1
  __shared__ __attribute__((aligned(16))) T s_row[2][W];       // the workgroup's best row, raw
  __shared__ __attribute__((aligned(16))) Cand s_c[2][NW];
  __shared__ __attribute__((aligned(16))) T s_grow[2][NW][W];  // the best row among a wavefront's records
  __shared__ __attribute__((aligned(16))) Cand s_g[2][NW];
  __shared__ T s_gr[2][NW];                                    // and its reciprocal
  __shared__ int s_ipiv[W];
  __shared__ T s_u12[W * LDU12];                               // pre: U12
  const int P = gridDim.x, g = blockIdx.x, t = threadIdx.x, lane = t & 63, e = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const long mp = m - j0;
  const long row0 = (long)g * ROWS;
  const int wr0 = wave * WR;   // the wavefront's first row

  // an earlier panel of this factorization failed: nothing to do (checked
  // after the loads below, which hide its latency)
  const unsigned failed = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // Rows travel between memory and LDS in 16-byte pieces, four lanes to one
  // row: lane i of a quad takes piece i of each of the quad's four rows in
  // turn, so a wavefront's access touches 16 rows x 64 bytes instead of 64
  // rows x 16 bytes (the panel's loads and stores took 17 us at 512 x 32
  // FP64 when every lane walked its own row).
  constexpr int NB = W / (4 * V);   // pieces of a row per lane
  const int li = lane & 3;
  auto load_rows = [&](long c0, vec (&v)[RPT][4][NB]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < RPT; q++)
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const long r = min(row0 + wr0 + q * 64 + (lane & ~3) + k, mp - 1);
        const T* src = At + c0 + (j0 + r) * ldt + li * V;
#pragma unroll
        for (int b = 0; b < NB; b++) v[q][k][b] = *(const vec*)(src + b * 4 * V);
      }
  };
  auto rows_to_lds = [&](const vec (&v)[RPT][4][NB]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < RPT; q++)
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int i = 0; i < V; i++)
            s_l[(b * 4 * V + li * V + i) * LDL + wr0 + q * 64 + (lane & ~3) + k] = v[q][k][b][i];
  };
  // a thread's own rows: y0 column j, up to date; y[k], k >= 2: column
  // j+k-1, which at the start of column j still lacks the update by column
  // j-1 (multiplier l, row j of s_u)
  T y0[RPT], y[RPT][W + 1], l[RPT];
  int pos[RPT];
  if (w == W) {
    vec v[RPT][4][NB];
    load_rows(j0, v);
    rows_to_lds(v);   // rows of this wavefront only
    wave_fence();
#pragma unroll
    for (int q = 0; q < RPT; q++) {
      y0[q] = s_l[wr0 + q * 64 + lane];
#pragma unroll
      for (int c = 1; c < W; c++) y[q][c + 1] = s_l[c * LDL + wr0 + q * 64 + lane];
    }
  } else {
#pragma unroll
    for (int q = 0; q < RPT; q++) {
      const T* src = At + j0 + (j0 + min(row0 + wr0 + q * 64 + lane, mp - 1)) * ldt;
      y0[q] = src[0];
#pragma unroll
      for (int c = 1; c < W; c++) {
        const T x = src[min(c, w - 1)];
        y[q][c + 1] = c < w ? x : T(0);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < RPT; q++) {
    const long r = row0 + wr0 + q * 64 + lane;
    pos[q] = r < mp ? (int)r : -1;
    y[q][0] = y[q][1] = T(0);
    l[q] = T(0);
  }
  if (failed) return;
  // pre: this panel is the right half of a 2W-wide node whose left half
  // [j0-W, j0) was just factored and its interchanges applied here.  The
  // node's TRSM and GEMM happen first: U12 = L11^{-1} A12 (every workgroup
  // solves the W x w block; workgroup 0 stores it at the end, after every
  // workgroup has read A12, which the first column's exchange guarantees),
  // then the rows lose L21 U12, on the matrix cores.
  if (pre) {
    vec v[RPT][4][NB];
    load_rows(j0 - W, v);   // the rows' multipliers, in flight during the solve
    __syncthreads();        // every wavefront has its rows in registers: s_l is free
    T* stg = s_l;           // L11 | A12: column j0-W+k of At, rows j0-W .. j0+W, at k*2W
    for (int i = t; i < W * 2 * W; i += L3_NT) {
      const int k = i / (2 * W), r = i % (2 * W);
      const T x = At[(j0 - W + min(r, W + w - 1)) + (j0 - W + k) * ldt];
      stg[i] = r < W + w ? x : T(0);
    }
    __syncthreads();
    if (t < W) {   // column t of U12: forward substitution with unit L11, a solved entry leaving all later ones at once
      T u[W];
#pragma unroll
      for (int k = 0; k < W; k++) u[k] = stg[k * 2 * W + W + t];
#pragma unroll
      for (int k = 0; k < W; k++) {
#pragma unroll
        for (int i = k + 1; i < W; i++) u[i] = lu_fms(stg[i * 2 * W + k], u[k], u[i]);
      }
#pragma unroll
      for (int k = 0; k < W; k++) s_u12[k * LDU12 + t] = u[k];
    }
    __syncthreads();
    rows_to_lds(v);
    wave_fence();
    // 16-row tiles of this wavefront: the multipliers are replaced by the
    // products, which every thread then subtracts from its own rows
    const int lr = lane & 15, lk = lane >> 4;
    T fb[2][W / 4];
#pragma unroll
    for (int n = 0; n < 2; n++)
#pragma unroll
      for (int k = 0; k < W / 4; k++) fb[n][k] = s_u12[(4 * k + lk) * LDU12 + 16 * n + lr];
#pragma unroll 1
    for (int i = 0; i < WR / 16; i++) {
      T* const tile = s_l + wr0 + 16 * i + lr;
      T fa[W / 4];
#pragma unroll
      for (int k = 0; k < W / 4; k++) fa[k] = tile[(4 * k + lk) * LDL];
      typename MF<T>::acc acc[2] = {};
#pragma unroll
      for (int k = 0; k < W / 4; k++)
#pragma unroll
        for (int n = 0; n < 2; n++) acc[n] = MF<T>::mma(fb[n][k], fa[k], acc[n]);
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int x = 0; x < 4; x++) tile[(16 * n + MF<T>::orow(lane, x)) * LDL] = acc[n][x];
    }
    wave_fence();
#pragma unroll
    for (int q = 0; q < RPT; q++) {
      y0[q] -= s_l[wr0 + q * 64 + lane];
#pragma unroll
      for (int c = 1; c < W; c++) y[q][c + 1] -= s_l[c * LDL + wr0 + q * 64 + lane];
    }
  }
  for (int i = t; i < (W + 1) * LDU; i += L3_NT) s_u[i] = T(0);   // no update before column 0, zeros past a row's end
  if constexpr (MULTI) {   // the next panel's records start empty
    for (int i = g * L3_NT + t; i < W * P * R::N; i += P * L3_NT) {
      const int c = i / (P * R::N), o = i % (P * R::N);
      wt_store(rec_next + c * R::COL + o, L3_EMPTY);
    }
  }
  __syncthreads();
  int stop = 0;
  // one wavefront of workgroup 0 keeps what the host and the interchange
  // kernels want to know, a column late, while the others wait for records:
  // the first zero pivot, and the rows that moved (lane i < w follows the row
  // that was at position i, lane 32+j the one first found at the pivot
  // position of column j when that lies past the panel's first w rows)
  int zinfo = 0, morig = lane < w ? lane : -1, mcur = morig, gprev = 0;
  T zprev = T(1);
  const bool keeper = g == 0 && wave == NW - 1;
  auto keep = [&](int j) __attribute__((always_inline)) {
    zinfo = (l3_rlf(zprev, 0) == T(0) && zinfo == 0) ? (int)(j0 + j + 1) : zinfo;
    const bool fresh = gprev >= w && __ballot(morig == gprev) == 0;
    if (fresh && lane == 32 + j) morig = mcur = gprev;
    mcur = mcur == gprev ? j : (mcur == j ? gprev : mcur);
  };
#pragma unroll 1
  for (int j = 0; j < w; j++) {
    const int buf = j & 1;
    // (a) the wavefront's best key and position to LDS; every lane already
    // takes the reciprocal of its own candidate, beside the reduction's chain
    KU key;
    unsigned np;
    bool second;
    T yb;
    {
      const bool v0 = pos[0] >= j, v1 = pos[1] >= j;
      const KU k0 = v0 ? LuKey<T>::key(y0[0], pos[0] == j) : KU(0), k1 = v1 ? LuKey<T>::key(y0[1], pos[1] == j) : KU(0);
      const unsigned n0 = v0 ? ~(unsigned)pos[0] : 0u, n1 = v1 ? ~(unsigned)pos[1] : 0u;
      second = (k1 > k0) | ((k1 == k0) & (n1 > n0));
      key = second ? k1 : k0;
      np = second ? n1 : n0;
      yb = second ? y0[1] : y0[0];
    }
    T rinv = (yb != T(0) && fabs(yb) >= MinNormal<T>::v) ? T(1) / yb : T(1);
    const int win = l3_best_lane(key, np);
    if (lane == win) {
      Cand cd;
      cd.key = key;
      cd.npos = np;
      s_c[buf][wave] = cd;
    }
    __syncthreads();
    // (b) the workgroup's best
    Cand best;
    int bw = 0;
    {
      Cand cc[NW];
#pragma unroll
      for (int v = 0; v < NW; v++) cc[v] = s_c[buf][v];
      best = cc[0];
#pragma unroll
      for (int v = 1; v < NW; v++) {
        const bool tk = cc[v].beats(best);
        best.key = tk ? cc[v].key : best.key;
        best.npos = tk ? cc[v].npos : best.npos;
        bw = tk ? v : bw;
      }
    }
    unsigned long long* recs = rec + (size_t)j * R::COL;
    if (wave == __builtin_amdgcn_readfirstlane(bw)) {
      // its wavefront lays the row out across the lanes (through LDS), adds
      // the update by column j-1 and publishes it
      const bool sec = (__ballot(second) >> win) & 1;
      auto put = [&](const T (&yy)[W + 1], T yy0) __attribute__((always_inline)) {
        T* dst = s_row[buf];
        dst[0] = yy0;
#pragma unroll
        for (int c = 1; c < W; c++) dst[c] = yy[c + 1];
      };
      T lb;
      if (sec) {
        lb = l3_rlf(l[1], win);
        if (lane == win) put(y[1], y0[1]);
      } else {
        lb = l3_rlf(l[0], win);
        if (lane == win) put(y[0], y0[0]);
      }
      wave_fence();
      rinv = l3_rlf(rinv, win);
      if constexpr (MULTI) {
        unsigned long long* dst = recs + (size_t)g * R::N;
        unsigned long long wd;
        bool need;
        int at;
        if constexpr (sizeof(T) == 8) {
          T v = s_row[buf][e];
          const T up = s_u[j * LDU + e + 1];
          v = e >= 1 ? lu_fms(lb, up, v) : v;
          // lanes 0..31 the row, 32 the position, 33 the reciprocal
          v = lane == 33 ? rinv : v;
          wd = (unsigned long long)__double_as_longlong(v);
          if (lane == 32) wd = (unsigned long long)best.npos << 32;
          need = lane < W - j || (lane & ~1) == 32;
          at = lane < 32 ? R::HW + lane : lane - 32;
        } else {
          const int e2 = 2 * (lane & 15);
          float a = s_row[buf][e2], b = s_row[buf][e2 + 1];
          const float ua = s_u[j * LDU + e2 + 1], ub = s_u[j * LDU + e2 + 2];
          a = e2 >= 1 ? lu_fms(lb, ua, a) : a;
          b = lu_fms(lb, ub, b);
          // lanes 0..15 the row, 16 position and reciprocal
          a = lane == 16 ? rinv : a;
          const unsigned hi = lane == 16 ? best.npos : __float_as_uint(b);
          wd = ((unsigned long long)hi << 32) | __float_as_uint(a);
          need = 2 * lane < W - j || lane == 16;
          need = need && lane <= 16;
          at = lane < 16 ? R::HW + lane : 0;
        }
        wd = wd == L3_EMPTY ? wd ^ 1 : wd;   // a NaN with another payload
        if (need) wt_store(dst + at, wd);
      } else {
        T v = s_row[buf][e];
        const T up = s_u[j * LDU + e + 1];
        v = e >= 1 ? lu_fms(lb, up, v) : v;
        if (lane < W) s_grow[buf][0][lane] = v;
        if (lane == 0) s_gr[buf][0] = rinv;
      }
    }
    // (c) the deferred update by column j-1, shifting every row by one
    // element, while the records travel
    {
      const T* u = s_u + j * LDU;
#pragma unroll
      for (int k0 = 0; k0 < W; k0 += 8) {
        T uk[8];
#pragma unroll
        for (int k = 0; k < 8; k++) uk[k] = u[k0 + k + 1];
#pragma unroll
        for (int k = k0 == 0 ? 1 : 0; k < 8; k++)
#pragma unroll
          for (int q = 0; q < RPT; q++) {
            y[q][k0 + k] = lu_fms(l[q], uk[k], y[q][k0 + k + 1]);
            asm volatile("" : "+v"(y[q][k0 + k]));   // in this order: each element into its own register
          }
      }
    }
    if (keeper && j > 0) keep(j - 1);
    T val;
    if constexpr (MULTI) {
      // (d) this wavefront's share of the records: wave, wave + NW, ...
      const int nrec = (P - wave + NW - 1) / NW;
      Cand wb;
      wb.key = 0;
      wb.npos = 0;
      T wr_inv = T(1);
      if (nrec > 0) {
        unsigned long long wd[NL], wk, wp, wi = 0;
        const int d = lane % R::RW, h = lane / R::RW;
        const bool need = d * 8 / (int)sizeof(T) < W - j;
        const unsigned long long* hsrc = recs + (size_t)(wave + NW * min(lane % NR, nrec - 1)) * R::N;
        int spins = 0;
        while (true) {
          wp = bypass_load(hsrc);
          if constexpr (sizeof(T) == 8) wi = bypass_load(hsrc + 1);
          wk = bypass_load(hsrc + R::HW);
#pragma unroll
          for (int i = 0; i < NL; i++) wd[i] = 0;
          if (need) {
#pragma unroll
            for (int i = 0; i < NL; i++)
              if (i * RPI < nrec) wd[i] = bypass_load(recs + (size_t)(wave + NW * min(i * RPI + h, nrec - 1)) * R::N + R::HW + d);
          }
          bool ok = (wp != L3_EMPTY) & (wk != L3_EMPTY) & (wi != L3_EMPTY);
#pragma unroll
          for (int i = 0; i < NL; i++) ok &= wd[i] != L3_EMPTY;
          if (__all(ok)) break;
          if (++spins > (1 << 22)) break;
        }
        T v0, rv;
        unsigned n;
        if constexpr (sizeof(T) == 8) {
          v0 = __longlong_as_double((long long)wk);
          rv = __longlong_as_double((long long)wi);
        } else {
          v0 = __uint_as_float((unsigned)wk);
          rv = __uint_as_float((unsigned)wp);
        }
        n = lane < nrec ? (unsigned)(wp >> 32) : 0u;
        const KU k = n != 0u ? LuKey<T>::key(v0, ~n == (unsigned)j) : KU(0);
        const int wr = l3_best_lane(k, n);
        wb.key = l3_rl(k, wr);
        wb.npos = spins > (1 << 22) ? FAIL : l3_rl(n, wr);
        wr_inv = l3_rlf(rv, wr);
        unsigned long long row = wd[0];
#pragma unroll
        for (int i = 1; i < NL; i++) row = (wr / RPI == i) ? wd[i] : row;
        if (h == wr % RPI) *(unsigned long long*)&s_grow[buf][wave][d * 8 / (int)sizeof(T)] = row;
      }
      if (lane == 0) {
        s_g[buf][wave] = wb;
        s_gr[buf][wave] = wr_inv;
      }
      __syncthreads();
      T cv[NW], cr[NW];
      Cand cc[NW];
#pragma unroll
      for (int v = 0; v < NW; v++) { cc[v] = s_g[buf][v]; cv[v] = s_grow[buf][v][e]; cr[v] = s_gr[buf][v]; }
      best = cc[0];
      val = cv[0];
      rinv = cr[0];
      bool bad = cc[0].npos == FAIL;
#pragma unroll
      for (int v = 1; v < NW; v++) {
        const bool tk = cc[v].beats(best);
        bad |= cc[v].npos == FAIL;
        best.key = tk ? cc[v].key : best.key;
        best.npos = tk ? cc[v].npos : best.npos;
        val = tk ? cv[v] : val;
        rinv = tk ? cr[v] : rinv;
      }
      const unsigned fp = ~best.npos;
      stop = __builtin_amdgcn_readfirstlane(bad ? 1 : (fp < (unsigned)j || fp >= (unsigned long)mp) ? 2 : 0);
      if (stop) break;
    } else {
      __syncthreads();
      val = s_grow[buf][0][e];
      rinv = s_gr[buf][0];
    }
    // (e) interchange (positions), multipliers, the next column
    const int gp = (int)__builtin_amdgcn_readfirstlane(~best.npos);
    const T u1 = l3_rlf(val, 1);
#pragma unroll
    for (int q = 0; q < RPT; q++) {
      pos[q] = pos[q] == gp ? j : (pos[q] == j ? gp : pos[q]);
      l[q] = y0[q] * rinv;
      s_l[j * LDL + wr0 + q * 64 + lane] = l[q];
      y0[q] = lu_fms(l[q], u1, y[q][1]);
    }
    if (wave == 0) {
      if (lane < 32) s_u[(j + 1) * LDU + lane] = val;
      if (lane == 0) s_ipiv[j] = gp;
    }
    gprev = gp;
    zprev = val;
  }
  if (stop) {
    if (t == 0) atomicExch(err, (unsigned)stop);
    return;
  }
  __syncthreads();   // the last row of s_u
  // Every row to its final position.  A pivot row (few, so by its own thread):
  // multipliers left of the diagonal, then its row of U.
#pragma unroll
  for (int q = 0; q < RPT; q++) {
    if (pos[q] < 0 || (pos[q] >= w && w == W)) continue;
    T* dst = At + j0 + (j0 + pos[q]) * ldt;
#pragma unroll
    for (int c = 0; c < W; c++) {
      const T x = pos[q] < w && c >= pos[q] ? s_u[(pos[q] + 1) * LDU + c - pos[q]] : s_l[c * LDL + wr0 + q * 64 + lane];
      if (c < w) dst[c] = x;
    }
  }
  if (w == W) {
#pragma unroll
    for (int q = 0; q < RPT; q++) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        // the position of the quad's row k
        const int p = k == 0   ? __builtin_amdgcn_update_dpp(0, pos[q], 0x00, 0xF, 0xF, false)
                      : k == 1 ? __builtin_amdgcn_update_dpp(0, pos[q], 0x55, 0xF, 0xF, false)
                      : k == 2 ? __builtin_amdgcn_update_dpp(0, pos[q], 0xAA, 0xF, 0xF, false)
                               : __builtin_amdgcn_update_dpp(0, pos[q], 0xFF, 0xF, 0xF, false);
        vec v[NB];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int i = 0; i < V; i++)
            v[b][i] = s_l[(b * 4 * V + li * V + i) * LDL + wr0 + q * 64 + (lane & ~3) + k];
        if (p >= w) {
          T* dst = At + j0 + (j0 + p) * ldt + li * V;
#pragma unroll
          for (int b = 0; b < NB; b++) *(vec*)(dst + b * 4 * V) = v[b];
        }
      }
    }
  }
  if (pre && g == 0) {
    for (int i = t; i < W * w; i += L3_NT) {
      const int k = i / w, c = i % w;
      At[(j0 + c) + (j0 - W + k) * ldt] = s_u12[k * LDU12 + c];
    }
  }
  if (keeper) {
    keep(w - 1);
    if (lane < w) ipiv[j0 + lane] = (int)(j0 + s_ipiv[lane] + 1);
    if (lane == 0 && zinfo != 0 && *info == 0) *info = zinfo;
    // the list of the rows that moved
    const bool mv = morig != mcur;
    const unsigned long long mm = __ballot(mv);
    if (mv) {
      const int k = __popcll(mm & ((1ull << lane) - 1));
      moves[1 + 2 * k] = mcur;
      moves[2 + 2 * k] = morig;
    }
    if (lane == 0) moves[0] = __popcll(mm);
  }
}
