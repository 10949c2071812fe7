// FP32 inner iterations of the batched MsFEM solve on the matrix cores.
// Included by msfem.hip inside its anonymous namespace, after Cell, SolveArgs
// and the stencil tables.
//
// One task holds NR right-hand sides of a cell (all 24 for cells of up to 384
// interior nodes, 12 for up to 768; 8 or 12 in batches too small to fill the
// chip so, see mfma_batch_rhs).  The stencil product q = K p is a 3x3
// block per (node, stencil point) times 3 x NR values, and every node has
// blocks of its own, so the product maps onto v_mfma_f32_4x4x1_16b_f32: 16
// independent 4x4 outer products.  Block = node (16 consecutive nodes per
// wave and instruction), rows = the 3 components (row 3 is not used),
// columns = 4 right-hand sides.  Per stencil point and component b a lane
// supplies K[a][b] of its node (a = lane % 4) and C = NR / 4 right-hand
// sides of p_b, for C instructions; column c = lane % 4 carries right-hand
// sides C c .. C c + C - 1.  An instruction covers 3 x 64 multiply-adds in 8
// cycles of a SIMD's matrix core, 12 on its FP32 vector unit.
//
// What else it buys: one task per cell instead of three reads K once per
// iteration for all 24 right-hand sides, and the three barriers and the
// scalar work of an iteration are shared by them too.  (With one task per
// cell nothing shares K in L2: 32 cells at a time hold 6.5 MB of it, an XCD's
// L2 4 MB, so K comes from the fabric in every iteration.)
//
// K is stored for it in lane order (k32_tile_index).  Lanes with
// lane % 4 == 3 read their neighbour's 16 bytes again.
//
// Bound and measurements (8^3 cells, one workgroup per CU, core cycles per
// iteration of a cell): the product took 14,200, against 13,000 of MFMA
// issue on the fullest SIMD; the update 5,100, the two reductions 8,500, the
// new direction 3,400; the FP64 sums of single products have since added
// about 1,200.  No unit is saturated over a launch (matrix cores busy 25 %,
// vector issue 35 %, LDS 38 %; a wave waits 46 % of its time): the phases
// follow each other behind barriers.  An FP64 residual pass costs as much as
// 4 to 7 iterations (K64 comes from HBM, twice).  32,768 cells of 8^3 from
// zero: 160 ms, against 215 ms for the one-row-per-thread vector kernel it
// replaces and 490 ms for the slab kernel (2 rows per thread) that untuned
// calls ran; 16^3 cells of n = 6..10: 29.1 against 85.1 ms.
//
// What decided it, one at a time at 4,096 cells of 8^3: everything in
// registers, spilled d 38.9 ms; half of d in LDS, addresses formed where they
// are used 26.2 (a spilled value reloaded in the loop waits for every K load
// in flight); p read two entries ahead of its use 24.7 (the compiler's own
// order waited for each read); three K64 points in flight 23.8.  Slower: K
// stored as its upper half, the lower blocks transposed by lane moves
// (32.1 ms: a third less traffic beyond L2, but 126 more vector instructions
// per 16 nodes); two workgroups of 4 waves with 12 right-hand sides per CU
// (38.1 ms: K is read twice).  Inner products added in FP32 per node first
// were 4 % faster (17.1 against 17.8 ms) and are not used.

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// right-hand sides per lane whose correction lives in LDS
constexpr int mfma_d_lds(int nr) { return nr == 24 ? 3 : nr == 12 ? 1 : 0; }
// Right-hand sides per task of a cell: all 24 while r, q and half of d of 24
// groups of 16 nodes fit the registers of 8 waves (n <= 8), else 12 (n = 9,
// 10: up to 48 groups).
__host__ __device__ constexpr int mfma_task_rhs(int nint) { return nint <= 384 ? 24 : 12; }

// Time of a cell's task in units of about 0.3 us of a batch of its own: each
// iteration costs a fixed part and one per node, and iterations grow with n.
// (24 right-hand sides, n = 3..8: 0.13 0.17 0.21 0.38 0.65 0.98 ms.)
inline int64_t mfma_task_weight(int n, int nint) { return 400 + (int64_t)n * nint; }
// Right-hand sides per task of a whole batch (0: mfma_task_rhs of each cell).
// A cell's wider tasks do less work in all (K is read once, the barriers are
// shared), narrower ones end sooner: 8^3 0.98 / 0.64 / 0.46 ms with 24 / 12 /
// 8, 5^3 0.21 / 0.16 / 0.12, 10^3 1.41 with 12, 1.00 with 8.  So the narrowest
// width is taken whose tasks, counted as fractions of the largest cell's, all
// run at once, one per CU: 85 cells of 8^3 1.08 -> 0.54 ms, 128 cells 1.11 ->
// 0.75; with 100 cells 8 at a time would take a second turn (0.99 ms, 12: 0.73).
inline int mfma_batch_rhs(int64_t weights, int64_t largest, int cus) {
  for (int nr : {8, 12})
    if (weights * (24 / nr) <= (int64_t)cus * largest) return nr;
  return 0;
}

struct MfmaRhs {  // per right-hand side of the running task
  double bb[NB], rr64[NB], prev[NB], scale[NB], itol2[NB];
  double rz[2][NB], rzkeep[NB], rrpred[NB], rrmin[2][NB], ratio[NB];
  int itmin[2][NB], done[NB], failed[NB], warm[NB], itbase[NB], it[NB];
};

// Workgroup sums of C values per lane (v[j] of right-hand side C c + j) over
// the 16 blocks of a wave and over the waves, in two steps: mfma_wave_sums
// leaves the wave's sums in part[wave][j][c], and after a barrier
// mfma_total of lane r < 4 C is the total of right-hand side r (the same in
// every wave).  The halves of a wave share the work of the last steps when C
// is even.
template <int C>
__device__ __forceinline__ void mfma_wave_sums(const double (&v)[C], double* part) {
  constexpr bool split = C % 2 == 0;
  constexpr int N = split ? C / 2 : C;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double a[N];
#pragma unroll
  for (int i = 0; i < N; i++) {
    a[i] = swap_add<32>(v[i], split ? v[N + i] : v[i]);
    a[i] = swap_add<16>(a[i], a[i]);
    a[i] += row_rotated<0x128>(a[i]);
    a[i] += row_rotated<0x124>(a[i]);
  }
  if ((lane & 28) == 0 && (split || lane < 32))
#pragma unroll
    for (int i = 0; i < N; i++) part[(wave * C + (split ? (lane >> 5) * N : 0) + i) * 4 + (lane & 3)] = a[i];
}
template <int C, int W>
__device__ __forceinline__ double mfma_total(const double* part, int r) {
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < W; w++) s += part[(w * C + r % C) * 4 + r / C];
  return s;
}

// q = K p for this wave's groups of 16 nodes (ngw of the G slots), and the
// per-lane partials of p.q.  K entries stream through a ring of PF chunks
// that wraps into the next product (K is the same): kr holds chunks 0 .. PF-1
// of the wave's first group on entry and on return.
constexpr int MF_PF = 4;
struct MfmaK {
  __amdgpu_buffer_rsrc_t rs;
  int vo;  // this lane's byte offset inside a chunk
  __device__ __forceinline__ f32x4_t at(int group, int chunk) const {
    return __builtin_bit_cast(f32x4_t,
                              __builtin_amdgcn_raw_buffer_load_b128(rs, vo, (group * KT_CHUNKS + chunk) * 768, 0));
  }
};

// The row and the strides that a product's addresses are formed from are made
// opaque to the compiler each time: otherwise it forms the addresses of all
// stencil points of all groups once per task and spills them.
__device__ __forceinline__ int opaque_s(int x) {
  asm volatile("" : "+s"(x));
  return x;
}
__device__ __forceinline__ int opaque_v(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

template <int NR, int G, int W>
__device__ __forceinline__ void mfma_product(const MfmaK& K, f32x4_t (&kr)[MF_PF], const float* P, int nint, int m,
                                             int wave, int blk, int c, int ngw, f32x4_t (&Q)[G][NR / 4],
                                             double (&w)[NR / 4]) {
  constexpr int C = NR / 4;
  static_assert(KT_CHUNKS % MF_PF == 0, "the ring's slots repeat per group");
#pragma unroll
  for (int g = 0; g < G; g++) {
    if (g < ngw) {
      const int grp = wave + W * g;
      const int gnext = g + 1 < ngw ? grp + W : wave;  // whose first chunks follow
      const int v = 16 * grp + opaque_v(blk);
      const int vi = min(v, nint - 1), mo = opaque_s(m);
#pragma unroll
      for (int j = 0; j < C; j++) Q[g][j] = f32x4_t{0, 0, 0, 0};
      // p from LDS PD entries ahead (an entry's C products take 8 C cycles, an
      // LDS read about 130); the scheduling barriers keep it that way
      constexpr int PD = C >= 6 ? 2 : C >= 3 ? 4 : 8;
      float pv[PD + 1][C];
      const float* pu[2];
      auto request = [&](int t) {
        const int s = t / 3, b = t % 3;
        if (b == 0) pu[s % 2] = P + neighbour_row(vi, stencil_offset(s, mo), nint) * (3 * NR) + C * c;
#pragma unroll
        for (int j = 0; j < C; j++) pv[t % (PD + 1)][j] = pu[s % 2][b * NR + j];
      };
#pragma unroll
      for (int t = 0; t < PD; t++) request(t);
#pragma unroll
      for (int t = 0; t < 3 * NS; t++) {
        if (t + PD < 3 * NS) request(t + PD);
        __builtin_amdgcn_sched_barrier(0);
        const float kv = kr[(t / 4) % MF_PF][t % 4];
#pragma unroll
        for (int j = 0; j < C; j++)
          Q[g][j] = __builtin_amdgcn_mfma_f32_4x4x1f32(kv, pv[t % (PD + 1)][j], Q[g][j], 0, 0, 0);
        if (t % 4 == 3 || t == 3 * NS - 1) {
          const int nx = t / 4 + MF_PF;
          kr[(t / 4) % MF_PF] = nx < KT_CHUNKS ? K.at(grp, nx) : K.at(gnext, nx - KT_CHUNKS);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int v = 16 * (wave + W * g) + opaque_v(blk);
    if (v < nint) {
      const float* pp = P + v * (3 * NR) + C * c;
#pragma unroll
      for (int j = 0; j < C; j++)
#pragma unroll
        for (int a = 0; a < 3; a++) w[j] += (double)(Q[g][j][a] * pp[a * NR + j]);
    }
  }
}

// One task: right-hand sides q0 .. q0 + NR - 1 of a cell.  In LDS: P
// [nint][3][NR] floats (16-byte aligned), behind it DL (part of the correction
// d) and DV, the FP32 inverse diagonal [nint][3].
// The algorithm, its stop tests and the continuation across FP64 residual
// replacements are those of k_batch_solve; lane r < NR of every wave decides
// for right-hand side r, wave 0 writes the state.
template <int NR, int G, int W>
__device__ __forceinline__ void mfma_task(const SolveArgs& A, const Cell& C_, int cell, int q0, float* P, float* DV, float* DL,
                                          double* partA, double* partB, MfmaRhs& S) {
  constexpr int C = NR / 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 3, blk = lane >> 2;
  const int n = C_.n, m = n - 1, nint = C_.nint;
  const int ng = mfma_groups(nint);
  const int ngw = wave < ng ? (ng - wave + W - 1) / W : 0;
  const double* K64 = A.K64 + C_.int0 * (NS * 9);
  const double* b64 = A.b64 + C_.int0 * (3 * NB) + q0;
  double* x64 = A.x64 + C_.int0 * (3 * NB) + q0;
  auto at64 = [&](int v, int a, int j) { return (unsigned)(v * (3 * NB) + a * NB + C * c + j); };
  MfmaK K;
  K.rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A.K32 + C_.kt0), (short)0,
                                           (int)(k32_tile_floats(nint) * sizeof(float)), kBufferRsrcWord3);
  K.vo = (blk * 3 + min(c, 2)) * 16;
  const __amdgpu_buffer_rsrc_t rs64 = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(K64), (short)0,
                                                                        NS * 9 * nint * 8, kBufferRsrcWord3);
  for (int e = tid; e < 3 * nint; e += 64 * W) DV[e] = A.dinv32[C_.int0 * 3 + e];
  const int inner_cap = min(A.inner_cap, 20 * n + 60);
  constexpr int kStagWindow = 60;
  constexpr unsigned kAll = NR == 32 ? ~0u : (1u << NR) - 1;
  // this lane's node of group slot g (opaque: its addresses are formed where
  // they are used)
  auto row = [&](int g) { return 16 * (wave + W * g) + opaque_v(blk); };
  const bool mine_r = lane < NR;
  const int sl = mine_r ? lane : 0;

  // the correction d: right-hand sides j < DJ of every lane in LDS, the rest
  // in registers (all of it, beside r and q, is more than a wave has)
  constexpr int DJ = mfma_d_lds(NR);
  auto dl = [&](int v, int a, int j) -> float& { return DL[(v * 3 + a) * (4 * DJ) + c * DJ + j]; };
  float R[G][3][C], D[G][3][C - DJ];
  f32x4_t Q[G][C];
  // ||b||^2 per right-hand side; x = 0 without a guess
  {
    double w[C];
#pragma unroll
    for (int j = 0; j < C; j++) w[j] = 0;
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int v = row(g);
      if (v >= nint) continue;
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int j = 0; j < C; j++) {
          const double bv = b64[at64(v, a, j)];
          w[j] += bv * bv;
          if (!A.use_guess) {
            x64[at64(v, a, j)] = 0.0;
            R[g][a][j] = (float)bv;  // the first residual
          }
        }
    }
    mfma_wave_sums<C>(w, partA);
    __syncthreads();
    if (tid < NR) {
      const double bb = mfma_total<C, W>(partA, tid);
      S.bb[tid] = bb > 0 ? bb : 1.0;
      S.rr64[tid] = bb;
      S.done[tid] = S.failed[tid] = S.warm[tid] = S.it[tid] = 0;
      S.prev[tid] = 1e300;
      S.scale[tid] = 1.0;
    }
    __syncthreads();
  }
  bool guess_checked = !A.use_guess;
  for (int outer = 0; outer < 64; outer++) {
    // true residual b - K64 x64 (FP64), kept in R unscaled; from the zero
    // start it is b
    double rrl = 0.0;
    if (outer == 0 && !A.use_guess) {
      rrl = S.rr64[sl];
    } else {
      double w[C];
#pragma unroll
      for (int j = 0; j < C; j++) w[j] = 0;
      // the iterate is staged in the place of p and d (FP64: part of every
      // lane's right-hand sides at a time); p waits in registers (q and d are
      // not live here)
      float Ps[G][3][C];
#pragma unroll
      for (int g = 0; g < G; g++) {
        const int v = row(g);
        if (v < nint)
#pragma unroll
          for (int a = 0; a < 3; a++)
#pragma unroll
            for (int j = 0; j < C; j++) Ps[g][a][j] = P[v * (3 * NR) + a * NR + C * c + j];
      }
      auto part = [&](auto first, auto count) {
        constexpr int J0 = decltype(first)::value, H = decltype(count)::value, ROW = 12 * H;
        static_assert(8 * ROW <= 4 * (3 * NR + 12 * DJ), "a staged row fits in the place of p and d");
        double* XS = reinterpret_cast<double*>(P);
        __syncthreads();  // every wave is past its reads of this region
#pragma unroll
        for (int g = 0; g < G; g++) {
          const int v = row(g);
          if (v < nint)
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
              for (int j = 0; j < H; j++) XS[v * ROW + a * 4 * H + H * c + j] = x64[at64(v, a, J0 + j)];
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < G; g++) {
          if (g >= ngw) continue;
          const int v = row(g), vi = min(v, nint - 1);
          const int stride = 8 * nint;
          double acc[3][H];
#pragma unroll
          for (int a = 0; a < 3; a++)
#pragma unroll
            for (int j = 0; j < H; j++) acc[a][j] = 0;
          // K64 comes from HBM: three points in flight
          double kn[3][9];
#pragma unroll
          for (int q = 0; q < 3; q++)
#pragma unroll
            for (int e = 0; e < 9; e++) kn[q][e] = buffer_load_f64(rs64, 8 * vi, (9 * q + e) * stride);
#pragma unroll 1
          for (int s0 = 0; s0 < NS; s0 += 3) {
#pragma unroll
            for (int q = 0; q < 3; q++) {
              const int u = neighbour_row(vi, stencil_offset(s0 + q, m), nint);
#pragma unroll
              for (int b = 0; b < 3; b++)
#pragma unroll
                for (int j = 0; j < H; j++) {
                  const double xv = XS[u * ROW + b * 4 * H + H * c + j];
#pragma unroll
                  for (int a = 0; a < 3; a++) acc[a][j] += kn[q][3 * a + b] * xv;
                }
              const int next = min(s0 + q + 3, NS - 1) * 9;  // (past the last point: not used)
#pragma unroll
              for (int e = 0; e < 9; e++) kn[q][e] = buffer_load_f64(rs64, 8 * vi, (next + e) * stride);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
          if (v < nint)
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
              for (int j = 0; j < H; j++) {
                const double rv = b64[at64(v, a, J0 + j)] - acc[a][j];
                w[J0 + j] += rv * rv;
                R[g][a][J0 + j] = (float)rv;
              }
        }
      };
      constexpr int H0 = C / 2 + C % 2;
      part(std::integral_constant<int, 0>{}, std::integral_constant<int, H0>{});
      part(std::integral_constant<int, H0>{}, std::integral_constant<int, C - H0>{});
      __syncthreads();
#pragma unroll
      for (int g = 0; g < G; g++) {
        const int v = row(g);
        if (v < nint)
#pragma unroll
          for (int a = 0; a < 3; a++)
#pragma unroll
            for (int j = 0; j < C; j++) P[v * (3 * NR) + a * NR + C * c + j] = Ps[g][a][j];
      }
      mfma_wave_sums<C>(w, partB);
      __syncthreads();
      rrl = mfma_total<C, W>(partB, sl);
    }
    if (!guess_checked) {
      // a guess whose residual exceeds the zero guess's (= ||b||) is dropped
      guess_checked = true;
      const bool badl = mine_r && !(rrl <= S.bb[sl]);
      const unsigned bad = (unsigned)__ballot(badl) & kAll;
      if (bad) {
        const unsigned bl = bad >> (C * c);
#pragma unroll
        for (int g = 0; g < G; g++) {
          const int v = row(g);
          if (v >= nint) continue;
#pragma unroll
          for (int a = 0; a < 3; a++)
#pragma unroll
            for (int j = 0; j < C; j++)
              if ((bl >> j) & 1) {
                x64[at64(v, a, j)] = 0.0;
                R[g][a][j] = (float)b64[at64(v, a, j)];
              }
        }
        if (badl) rrl = S.bb[sl];
        if (wave == 0 && badl) A.flags[cell * NB + q0 + lane] |= 2;
      }
    }
    if (tid < NR) {
      const int r = tid;
      const double rr = rrl;
      // an outer step that did not reduce the true residual means the inner
      // precision cannot solve this problem: stop it and report it
      int failed = S.failed[r], done = S.done[r], warm = S.warm[r];
      if (!done && outer > 0 && !(rr < 0.9 * S.prev[r])) failed = 1;
      S.rr64[r] = rr;
      S.prev[r] = rr;
      // continue the FP32 iteration only if its recursion stayed consistent
      // with the true residual (within 2x in norm)
      if (warm && !(rr <= 4.0 * S.rrpred[r] * S.scale[r] * S.scale[r])) warm = 0;
      done = done || failed || (rr <= A.tol * A.tol * S.bb[r]) || !(rr == rr);
      S.failed[r] = failed;
      S.done[r] = done;
      S.warm[r] = warm;
      const double sc = rr > 0 ? sqrt(rr) : 1.0;
      S.ratio[r] = S.scale[r] / sc;
      S.scale[r] = sc;
      const double rel = sqrt(rr / S.bb[r]);
      const double it = fmin(fmax(A.inner_tol, 0.5 * A.tol / rel), 0.5);
      S.itol2[r] = it * it;
      S.itbase[r] = S.it[r];
    }
    __syncthreads();
    const bool livel = mine_r && !S.done[sl];
    const unsigned live = (unsigned)__ballot(livel) & kAll;
    if (!live || !__ballot(livel && S.it[sl] < A.maxit)) break;
    // start: R <- R/scale, D = 0, z = dinv R; the direction is z (fresh) or
    // z + beta ratio p_kept (continuation)
    unsigned act;
    {
      double w[C], w2[C];
#pragma unroll
      for (int j = 0; j < C; j++) w[j] = w2[j] = 0;
      float inv[C];
      const unsigned ll = live >> (C * c);
#pragma unroll
      for (int j = 0; j < C; j++) inv[j] = ((ll >> j) & 1) ? (float)(1.0 / S.scale[C * c + j]) : 0.f;
#pragma unroll
      for (int g = 0; g < G; g++) {
        const int v = row(g);
        if (v >= nint) continue;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const float dv = DV[3 * v + a];
#pragma unroll
          for (int j = 0; j < C; j++) {
            const float rv = ((ll >> j) & 1) ? (float)((double)R[g][a][j] * (double)inv[j]) : 0.f;
            R[g][a][j] = rv;
            if (j < DJ)
              dl(v, a, j) = 0;
            else
              D[g][a][j - DJ] = 0;
            const float z = dv * rv;
            w[j] += (double)(rv * z);
            w2[j] += (double)(rv * rv);
          }
        }
      }
      mfma_wave_sums<C>(w, partA);
      mfma_wave_sums<C>(w2, partA + 4 * C * W);
      __syncthreads();
      const double rz0 = mfma_total<C, W>(partA, sl), rr0 = mfma_total<C, W>(partA + 4 * C * W, sl);
      const bool on = livel && rr0 > S.itol2[sl];
      act = (unsigned)__ballot(on) & kAll;
      float be = 0.f;
      if (on && S.warm[sl] && S.rzkeep[sl] > 0.0 && S.ratio[sl] > 0.0) be = (float)(rz0 / (S.rzkeep[sl] * S.ratio[sl]));
      float beta[C];
#pragma unroll
      for (int j = 0; j < C; j++) beta[j] = __shfl(be, C * c + j, 64);
      if (tid < NR) {
        S.rz[0][tid] = rz0;
        S.rrmin[0][tid] = rr0;
        S.itmin[0][tid] = 0;
      }
#pragma unroll
      for (int g = 0; g < G; g++) {
        const int v = row(g);
        if (v >= nint) continue;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const float dv = DV[3 * v + a];
#pragma unroll
          for (int j = 0; j < C; j++) {
            float* pe = P + v * (3 * NR) + a * NR + C * c + j;
            const float z = dv * R[g][a][j];
            *pe = beta[j] != 0.f ? z + beta[j] * *pe : z;
          }
        }
      }
      __syncthreads();
    }
    int inner_it = 0, par = 0;
    unsigned capfail = 0;
    if (act && inner_cap > 0) {
      f32x4_t kr[MF_PF];
      if (ngw > 0)
#pragma unroll
        for (int q = 0; q < MF_PF; q++) kr[q] = K.at(wave, q);
      do {
        float alpha[C];
        {
          double w[C];
#pragma unroll
          for (int j = 0; j < C; j++) w[j] = 0;
          mfma_product<NR, G, W>(K, kr, P, nint, m, wave, blk, c, ngw, Q, w);
          const double rzp = S.rz[par][sl];
          mfma_wave_sums<C>(w, partB);
          __syncthreads();
          const double pq = mfma_total<C, W>(partB, sl);
          float al = 0.f;
          if (mine_r && ((act >> sl) & 1) && pq != 0.0) al = (float)(rzp / pq);
#pragma unroll
          for (int j = 0; j < C; j++) alpha[j] = __shfl(al, C * c + j, 64);
        }
        unsigned act2;
        float beta[C];
        {
          // d, r, r.z and r.r group by group; where q and d leave no registers
          // for both sums, r.r afterwards from the new r (8^3 cells 17.8 ms,
          // both at once 18.4; 10^3 cells 13.0 and 12.8, 6^3 4.50 and 4.38).
          // One conversion and FP64 products: 1.5 % less time than FP32
          // products converted one by one.
          constexpr bool both = NR < 24 || G < 3;
          double w[C], w2[C];
#pragma unroll
          for (int j = 0; j < C; j++) w[j] = w2[j] = 0;
#pragma unroll
          for (int g = 0; g < G; g++) {
            const int v = row(g);
            if (v >= nint) continue;
#pragma unroll
            for (int a = 0; a < 3; a++) {
              const double dvd = DV[3 * v + a];
#pragma unroll
              for (int j = 0; j < C; j++) {
                const float pe = P[v * (3 * NR) + a * NR + C * c + j];
                if (j < DJ)
                  dl(v, a, j) += alpha[j] * pe;
                else
                  D[g][a][j - DJ] += alpha[j] * pe;
                const float rv = R[g][a][j] - alpha[j] * Q[g][j][a];
                R[g][a][j] = rv;
                const double rd = rv, r2 = rd * rd;
                w[j] += r2 * dvd;
                if (both) w2[j] += r2;
              }
            }
          }
          mfma_wave_sums<C>(w, partA);
          if constexpr (!both) {
#pragma unroll
            for (int g = 0; g < G; g++) {
              if (row(g) >= nint) continue;
#pragma unroll
              for (int j = 0; j < C; j++)
#pragma unroll
                for (int a = 0; a < 3; a++) w2[j] += (double)R[g][a][j] * (double)R[g][a][j];
            }
          }
          mfma_wave_sums<C>(w2, partA + 4 * C * W);
          const double rz_old = S.rz[par][sl], itol2 = S.itol2[sl], rrmin = S.rrmin[par][sl];
          const int itbase = S.itbase[sl], itmin = S.itmin[par][sl];
          __syncthreads();
          const double rzl = mfma_total<C, W>(partA, sl), rr = mfma_total<C, W>(partA + 4 * C * W, sl);
          const bool on = mine_r && ((act >> sl) & 1);
          bool cont = false, stag = false;
          float be = 0.f;
          if (on) {
            const bool stop = !(rr == rr) || rr <= itol2 || itbase + inner_it + 1 >= A.maxit;
            if (!stop) {
              const int itm = rr < 0.25 * rrmin ? inner_it + 1 : itmin;
              stag = inner_it + 1 - itm > kStagWindow;
            }
            cont = !(stop || stag);
            if (cont) be = (float)(rzl / rz_old);
          }
          act2 = (unsigned)__ballot(cont) & kAll;
          capfail |= (unsigned)__ballot(stag) & kAll;  // recorded after the x update
#pragma unroll
          for (int j = 0; j < C; j++) beta[j] = __shfl(be, C * c + j, 64);
          if (tid < NR) {
            const bool mark = on && rr < 0.25 * rrmin;
            S.rrmin[par ^ 1][tid] = mark ? rr : rrmin;
            S.itmin[par ^ 1][tid] = mark ? inner_it + 1 : itmin;
            S.rz[par ^ 1][tid] = on && cont ? rzl : rz_old;
            if (on && !cont) {
              // stopped: keep (p, r.z) of this iteration for the next step
              S.rzkeep[tid] = rz_old;
              S.it[tid] = itbase + inner_it + 1;
              S.warm[tid] = rr <= itol2;
              S.rrpred[tid] = rr;
            }
          }
        }
        // p = z + beta p (continuing right-hand sides only)
        const unsigned al2 = act2 >> (C * c);
#pragma unroll
        for (int g = 0; g < G; g++) {
          const int v = row(g);
          if (v >= nint) continue;
#pragma unroll
          for (int a = 0; a < 3; a++) {
            const float dv = DV[3 * v + a];
#pragma unroll
            for (int j = 0; j < C; j++) {
              float* pe = P + v * (3 * NR) + a * NR + C * c + j;
              const float pn = dv * R[g][a][j] + beta[j] * *pe;
              *pe = ((al2 >> j) & 1) ? pn : *pe;
            }
          }
        }
        __syncthreads();
        act = act2;
        par ^= 1;
        inner_it++;
      } while (act && inner_it < inner_cap);
    }
    // right-hand sides still active here reached the iteration cap
    capfail |= act;
    // x64 += scale * d (not for problems whose inner solve failed)
    {
      const unsigned fl = (unsigned)__ballot(mine_r && S.failed[sl]) & kAll;
      const unsigned upd = (live & ~capfail & ~fl) >> (C * c);
      double sc[C];
#pragma unroll
      for (int j = 0; j < C; j++) sc[j] = S.scale[C * c + j];
#pragma unroll
      for (int g = 0; g < G; g++) {
        const int v = row(g);
        if (v >= nint) continue;
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
          for (int j = 0; j < C; j++)
            if ((upd >> j) & 1) x64[at64(v, a, j)] += sc[j] * (double)(j < DJ ? dl(v, a, j) : D[g][a][j - DJ]);
      }
    }
    __syncthreads();
    if (tid < NR && ((capfail >> tid) & 1)) {
      S.failed[tid] = 1;
      S.it[tid] = S.itbase[tid] + inner_it;
    }
    if (inner_it == 0) break;  // nothing more can be done
  }
  __syncthreads();
  if (tid < NR) {
    const int at = cell * NB + q0 + tid;
    A.iters[at] = S.it[tid];
    A.relres[at] = sqrt(S.rr64[tid] / S.bb[tid]);
    int f = 0;
    if (!(S.rr64[tid] <= A.tol * A.tol * S.bb[tid])) f |= 1;
    if (S.failed[tid]) f |= A.list_failures ? (4 | 8) : 4;
    if (f) A.flags[at] |= f;
  }
  __syncthreads();
}

// Launch classes by the batch's largest cell: 0: nint <= 64 and 1: nint <= 128
// (4 waves of 1 / 2 groups, several workgroups per CU), 2: nint <= 384 (8
// waves of up to 3 groups, one workgroup per CU: p and d take its LDS), 3:
// nint <= 729 (up to 6 groups; tasks of 24 and of 12 right-hand sides in one
// launch), 4: tasks of 8 with nint <= 512 (up to 4 groups: one cell of 9^3
// 0.68 -> 0.65 ms; the wider tasks gain nothing from it).
__host__ __device__ constexpr int mfma_class(int max_nint, int task_rhs) {
  return max_nint <= 64 ? 0 : max_nint <= 128 ? 1 : max_nint <= 384 ? 2 : max_nint <= 512 && task_rhs == 8 ? 4 : 3;
}
constexpr int mfma_waves(int cls) { return cls <= 1 ? 4 : 8; }
constexpr int mfma_eu(int cls) { return cls == 0 ? 3 : 2; }

// NRT: right-hand sides per task, 0 for mfma_task_rhs of the task's cell.
template <int CLS, int NRT>
__global__ __launch_bounds__(mfma_waves(CLS) * 64)
__attribute__((amdgpu_waves_per_eu(mfma_eu(CLS), mfma_eu(CLS))))
void k_batch_solve_mfma(SolveArgs A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int W = mfma_waves(CLS);
  __shared__ double partA[W * 12 * 4];
  __shared__ double partB[W * 6 * 4];
  __shared__ MfmaRhs S;
  __shared__ int task_s;
  float* P = reinterpret_cast<float*>(smem_raw);
  int tried = 0;  // queues found empty (thread 0)
  const int home = blockIdx.x % NQ;
  for (;;) {
    if (threadIdx.x == 0) {
      int t = -1;
      while (tried < NQ) {
        const int q = (home + tried) % NQ;
        const int k = (int)__hip_atomic_fetch_add(A.queue + q * QSTRIDE, 1u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
        if (A.seg[q] + k < A.seg[q + 1]) {
          t = A.seg[q] + k;
          break;
        }
        tried++;
      }
      task_s = t;
    }
    __syncthreads();
    const int task = __builtin_amdgcn_readfirstlane(task_s);
    if (task < 0) break;
    const int cell = __builtin_amdgcn_readfirstlane(A.task_cell[task]);
    const int grp = __builtin_amdgcn_readfirstlane(A.task_group[task]);
    const Cell C = uniform_cell(A.cells, cell);
    constexpr int G = CLS == 3 ? 6 : CLS == 4 ? 4 : CLS == 2 ? 3 : CLS + 1;
    if constexpr (NRT == 8) {
      mfma_task<8, G, W>(A, C, cell, 8 * grp, P, P + C.nint * 24, P, partA, partB, S);
    } else if constexpr (NRT == 12) {
      mfma_task<12, G, W>(A, C, cell, 12 * grp, P, P + C.nint * 48, P + C.nint * 36, partA, partB, S);
    } else if constexpr (CLS == 3) {
      if (C.nint > 384)
        mfma_task<12, G, W>(A, C, cell, 12 * grp, P, P + C.nint * 48, P + C.nint * 36, partA, partB, S);
      else
        mfma_task<24, 3, W>(A, C, cell, 0, P, P + C.nint * 108, P + C.nint * 72, partA, partB, S);
    } else {
      mfma_task<24, G, W>(A, C, cell, 0, P, P + C.nint * 108, P + C.nint * 72, partA, partB, S);
    }
  }
}

// The FP64 pass's task list: groups of RG right-hand sides of a cell with a
// problem that the FP32 launch handed over (flag bit 3).
__global__ void k_list_failures(const int* __restrict__ flags, int ngroups, int* fb_count, int* fb_cell,
                                int* fb_group) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ngroups) return;
  int any = 0;
#pragma unroll
  for (int r = 0; r < RG; r++) any |= flags[(int64_t)i * RG + r] & 8;
  if (any) {
    const int slot = __hip_atomic_fetch_add(fb_count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    fb_cell[slot] = i / (NB / RG);
    fb_group[slot] = i % (NB / RG);
  }
}
