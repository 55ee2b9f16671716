// Batched complex solve A X = B in few launches: blocked Gauss-Jordan with
// partial pivoting in product form, for orders up to GJ_MAX_N.
//
// The columns of A are taken in panels of 16.  Eliminating a panel's columns
// from every row (rows already used as pivots included) is one small matrix:
// with the panel's pivot rows p and G the n x 16 result of the elimination
//   strip[i] <- (i in p ? 0 : strip[i]) + G[i] strip[p]      for every column
// to the right and for B.  G of a panel (A11^-1 on its pivot rows, -A21 A11^-1
// elsewhere) overwrites the panel's columns of A, and `perm` keeps which row
// each column was eliminated with: rows are never moved, so nothing is
// interchanged, and X[k] is row perm[k] of the transformed B.
//
// gj_factor_kernel: 64, 128 or all columns in one launch, one workgroup per
//   system, a wavefront per 48 or 64 rows.  A panel's columns are loaded into MFMA
//   accumulators, the launch's earlier panels are applied to them (left-looking:
//   A is read and written once), and the panel is eliminated in registers, one
//   row per lane: a pivot step is one integer maximum over the lanes (DPP), one
//   LDS exchange of the pivot row and one barrier.
// gj_strips_kernel: one workgroup per system and strip of 16 CB columns, of B or
//   of the columns of A still to be factored.  The strip stays in MFMA
//   accumulators from its load to its store while the panels pass by: 8 n^2
//   operations per column on the matrix cores with B moved once; the 16 pivot
//   rows of a panel go through LDS, G comes from L2 (the strips of one system run
//   on one XCD).
// The multi-launch LU (lu_blocked.hip) needs 11 panel launches, as many trailing
// updates and 22 leaf launches for n = 162 and moves the trailing matrix once per
// panel.  Measured, LU -> here, ms: n = 50 (50 right-hand sides) 2 systems 0.28 ->
// 0.08, 4 096 systems 4.4 -> 0.42; n = 162 (162) 2 048 systems 7.0 -> 3.6; n = 338
// (338) 512 systems 11.1 -> 7.1, 2 systems (1.5 when one launch factored all
// columns) 0.89.  The solve runs at about 70 % of the FP64 matrix rate; the
// factorization is bound by the latency of its pivot steps (about 1 us: maximum,
// LDS exchange, barrier, reciprocal).
// Error: forward error as an LU's; the residual of an ill-conditioned system can
// be larger (Gauss-Jordan is not row-wise backward stable), so it serves the
// systems that are well conditioned by construction.
#include "khx_internal.h"
#include "khx_prof.h"

namespace khx {

namespace {

typedef double gj_d4 __attribute__((ext_vector_type(4)));
constexpr int NB = 16;      // panel width
constexpr int YS = NB + 1;  // LDS row stride

// maximum over the 64 lanes (DPP: inside rows of 16, then across the rows)
__device__ __forceinline__ int wave_max_int(int v) {
  int t;
#define GJ_STEP(ctrl, rmask)                                      \
  t = __builtin_amdgcn_update_dpp(v, v, ctrl, rmask, 0xf, false); \
  v = t > v ? t : v;
  GJ_STEP(0x111, 0xf)  // row_shr:1
  GJ_STEP(0x112, 0xf)  // row_shr:2
  GJ_STEP(0x114, 0xf)  // row_shr:4
  GJ_STEP(0x118, 0xf)  // row_shr:8
  GJ_STEP(0x142, 0xa)  // row_bcast:15
  GJ_STEP(0x143, 0xc)  // row_bcast:31
#undef GJ_STEP
  return __builtin_amdgcn_readlane(v, 63);
}

// 1 / v for any finite v: scaled by a power of two, Newton steps on the
// hardware's reciprocal, no branch (all lanes take it while the pivot search
// runs).  v = 0 gives NaN: the system is reported singular, its result is NaN.
__device__ __forceinline__ cd recip_pivot(cd v) {
  const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(v.x), fabs(v.y)));
  const double x = ldexp(v.x, -e), y = ldexp(v.y, -e);
  const double d = fma(x, x, y * y);
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  r = fma(r, fma(-d, r, 1.0), r);
  return mkc(ldexp(x * r, -e), ldexp(-y * r, -e));
}

// 16-byte aligned complex for LDS (one b128 access each)
struct alignas(16) lcd {
  double x, y;
};

// ------------------------------------------------------------ panel application
// A strip of 16 CB columns in MFMA accumulators: wavefront w holds rows
// 16 RB w .. + 16 RB, register r of lane l row l / 16 + 4 r of a block, column
// l % 16.  `slot` are the rows' places in the elimination order.
//
// One panel: the strip's pivot rows go to Y in LDS and leave the accumulators,
// then strip += G Y on the matrix cores.  The sixteen k of a panel are dealt so
// that a lane reads 64 adjacent bytes of its row of G (k = 4 (l / 16) + h, h = 0
// .. 3, one MFMA each).  G is fetched in two halves (h = 0, 1 and h = 2, 3),
// each one half ahead of its use.
template <int RB, int CB>
struct Strip {
  gj_d4 re[RB][CB], im[RB][CB];
  int slot[RB][4];
};

template <int RB>
struct Frag {
  cd v[RB][2];
};

// Offsets stay in 32 bits (zgj_solve checks).  Rows past n and columns past the
// last panel are read from the edge: their products go to rows that are never
// stored or meet zero rows of Y.
template <int RB>
__device__ __forceinline__ void fetch(Frag<RB>& f, const cd* __restrict__ a, const unsigned (&roff)[RB], int kcol,
                                      int last) {
  const unsigned c0 = (unsigned)min(kcol, last), c1 = (unsigned)min(kcol + 1, last);
#pragma unroll
  for (int t = 0; t < RB; ++t) {
    f.v[t][0] = a[roff[t] + c0];
    f.v[t][1] = a[roff[t] + c1];
  }
}

// (rows that are not the panel's go to the spare row NB: no branches)
template <int RB, int CB>
__device__ __forceinline__ void take_pivot_rows(Strip<RB, CB>& x, int first, lcd* Y, int li) {
  constexpr int YC = 16 * CB + 1;
#pragma unroll
  for (int t = 0; t < RB; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned s = min((unsigned)(x.slot[t][r] - first), (unsigned)NB);
      const bool mine = s < NB;
#pragma unroll
      for (int u = 0; u < CB; ++u) {
        Y[s * YC + u * 16 + li] = lcd{x.re[t][u][r], x.im[t][u][r]};
        x.re[t][u][r] = mine ? 0.0 : x.re[t][u][r];
        x.im[t][u][r] = mine ? 0.0 : x.im[t][u][r];
      }
    }
}

template <int RB, int CB, int H0>
__device__ __forceinline__ void multiply(Strip<RB, CB>& x, const Frag<RB>& f, const lcd* Y, int li, int lk, int blocks) {
  constexpr int YC = 16 * CB + 1;
  lcd bv[2][CB];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int u = 0; u < CB; ++u) bv[h][u] = Y[(4 * lk + H0 + h) * YC + u * 16 + li];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < RB; ++t) {
      if (t >= blocks) continue;  // uniform over the wavefront
      const cd av = f.v[t][h];
      const double nai = -av.y;
#pragma unroll
      for (int u = 0; u < CB; ++u) {
        x.re[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, bv[h][u].x, x.re[t][u], 0, 0, 0);
        x.im[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, bv[h][u].y, x.im[t][u], 0, 0, 0);
        x.re[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(nai, bv[h][u].y, x.re[t][u], 0, 0, 0);
        x.im[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, bv[h][u].x, x.im[t][u], 0, 0, 0);
      }
    }
}

// panels j0 .. j1 - 1 in order; Y: two buffers of 17 x (16 CB + 1); nbl: columns
// of panel j1 - 1
template <int RB, int CB>
__device__ __forceinline__ void apply_panels(Strip<RB, CB>& x, const cd* __restrict__ a, int lda, int n, int j0, int j1,
                                             int nbl, lcd* Y, int row0, int li, int lk) {
  constexpr int YC = 16 * CB + 1;
  if (j0 >= j1) return;
  const int left = n - row0, blocks = left <= 0 ? 0 : (left + 15) / 16;
  unsigned roff[RB];
#pragma unroll
  for (int t = 0; t < RB; ++t) roff[t] = (unsigned)(min(row0 + t * 16 + li, n - 1) * lda);
  Frag<RB> f0, f1;
  fetch(f0, a, roff, j0 * NB + 4 * lk, n - 1);
  for (int j = j0; j < j1; ++j) {
    lcd* y = Y + (j & 1) * (NB + 1) * YC;
    if (nbl < NB && j == j1 - 1)  // the rows that a narrower last panel does not have
      for (int e = threadIdx.x; e < (NB - nbl) * YC; e += blockDim.x) y[nbl * YC + e] = lcd{0.0, 0.0};
    take_pivot_rows(x, j * NB, y, li);
    fetch(f1, a, roff, j * NB + 4 * lk + 2, n - 1);
    __syncthreads();
    multiply<RB, CB, 0>(x, f0, y, li, lk, blocks);
    fetch(f0, a, roff, (j + 1) * NB + 4 * lk, n - 1);
    multiply<RB, CB, 2>(x, f1, y, li, lk, blocks);
  }
}

// ------------------------------------------------------------ factorization
// A wavefront's candidate for the pivot of a step.
struct Candidate {
  lcd row[NB];
  lcd recip;
};
constexpr int GJ_MAX_WAVES = 8;

// Columns c0 .. c1 - 1 (c0 a multiple of 16), to which the panels before c0 have
// been applied.  Workgroups of ceil(n / (16 RB)) wavefronts; in the elimination
// lane l of wavefront w owns row 16 RB w + l (l < 16 RB).
template <int RB>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(RB <= 3 ? 3 : 2))) void gj_factor_kernel(int n, int c0, int c1, cd* A, int lda, long long sA, int* perm, int* info) {
  extern __shared__ lcd sm[];
  const int nw = blockDim.x >> 6;
  lcd* stage = sm;                                                         // nw x 16 x YS, wavefront-private
  lcd* Y = stage + nw * 16 * YS;                                           // 2 x 17 x YS
  Candidate* cand = reinterpret_cast<Candidate*>(Y + 2 * (NB + 1) * YS);   // 2 x 8
  int4* keys = reinterpret_cast<int4*>(cand + 2 * GJ_MAX_WAVES);           // 2 x 8 (key, row) pairs
  int* ord = reinterpret_cast<int*>(keys + GJ_MAX_WAVES);                  // 16 RB nw
  const long long item = blockIdx.x;
  cd* a = A + item * sA;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int row0 = wave * 16 * RB;
  const int row = lane < 16 * RB ? row0 + lane : n;  // the row this lane eliminates
  int first_zero = 0;
  for (int e = tid; e < 16 * RB * nw; e += blockDim.x) ord[e] = 1 << 30;
  if (tid < GJ_MAX_WAVES) keys[tid] = make_int4(-2, 0, -2, 0);
  __syncthreads();
  for (int k = tid; k < c0; k += blockDim.x) ord[perm[item * n + k]] = k;
  __syncthreads();
  bool open = row < n && ord[min(row, n - 1)] == 1 << 30;
  for (int k0 = c0; k0 < c1; k0 += NB) {
    const int nb = min(NB, n - k0);
    cd x[NB];
    {
      // (rows past n and columns past the last panel's: the edge's values, which
      // reach nothing that is stored)
      Strip<RB, 1> st;
      const int gc = min(k0 + li, n - 1);
#pragma unroll
      for (int t = 0; t < RB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int gr = row0 + t * 16 + lk + 4 * r;
          const cd v = a[(unsigned)(min(gr, n - 1) * lda + gc)];
          st.re[t][0][r] = v.x;
          st.im[t][0][r] = v.y;
          st.slot[t][r] = ord[gr];
        }
      apply_panels(st, a, lda, n, c0 / NB, k0 / NB, NB, Y, row0, li, lk);
      // accumulators -> one row per lane, 16 rows at a time through the
      // wavefront's own LDS
      lcd* sp = stage + wave * 16 * YS;
#pragma unroll
      for (int c = 0; c < NB; ++c) x[c] = mkc(0.0, 0.0);
#pragma unroll
      for (int t = 0; t < RB; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sp[(lk + 4 * r) * YS + li] = lcd{st.re[t][0][r], st.im[t][0][r]};
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lk == t) {
#pragma unroll
          for (int c = 0; c < NB; ++c) x[c] = mkc(sp[li * YS + c].x, sp[li * YS + c].y);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
    // Eliminate the panel's columns.  The columns rotate through x: the current
    // one is x[0], the others move down by one as they are updated and the
    // finished column enters at the end, so one loop body serves every step and
    // sixteen steps restore the order.
    // key: the high word of |re| + |im| orders the candidates to 2^-20; rows
    // already used have -1
    int key = open ? __double2hiint(cabs1(x[0])) & 0x7fffffff : -1;
    cd rc = recip_pivot(x[0]);
    int best = wave_max_int(key);
#pragma unroll 1
    for (int jj = 0; jj < nb; ++jj) {
      const int buf = (jj & 1) * GJ_MAX_WAVES;
      const int src = __ffsll((unsigned long long)__ballot(key == best)) - 1;
      if (lane == src) {
        Candidate& c = cand[buf + wave];
        reinterpret_cast<int2*>(keys)[buf + wave] = make_int2(best, row);
#pragma unroll
        for (int q = 0; q < NB; ++q) c.row[q] = lcd{x[q].x, x[q].y};
        c.recip = lcd{rc.x, rc.y};
      }
      __syncthreads();
      int w = 0, kbest = best, prow = row0 + src;
      if (nw > 1) {
        int4 kq[GJ_MAX_WAVES / 2];
#pragma unroll
        for (int q = 0; q < GJ_MAX_WAVES / 2; ++q) kq[q] = keys[buf / 2 + q];
        kbest = kq[0].x;
        prow = kq[0].y;
#pragma unroll
        for (int q = 1; q < GJ_MAX_WAVES; ++q) {
          const int k = q & 1 ? kq[q / 2].z : kq[q / 2].x, r = q & 1 ? kq[q / 2].w : kq[q / 2].y;
          const bool more = k > kbest;
          w = more ? q : w;
          prow = more ? r : prow;
          kbest = more ? k : kbest;
        }
        w = __builtin_amdgcn_readfirstlane(w);
      }
      const Candidate& c = cand[buf + w];
      const lcd rp = c.recip;
      lcd pa[8], pb[7];
#pragma unroll
      for (int q = 0; q < 8; ++q) pa[q] = c.row[q + 1];
      __builtin_amdgcn_sched_barrier(0);  // half of the row is on its way before the first use
      if (kbest == 0 && first_zero == 0) first_zero = k0 + jj + 1;
      cd m = x[0] * mkc(rp.x, rp.y);
      if (row == prow) {
        open = false;
        ord[row] = k0 + jj;
        m = mkc(-rp.x, -rp.y);
#pragma unroll
        for (int q = 0; q < NB; ++q) x[q] = mkc(0.0, 0.0);
      }
      // the next column first: its pivot search and reciprocals run beside the
      // other columns' updates
      x[0] = fmsc(x[1], m, mkc(pa[0].x, pa[0].y));
      key = open ? __double2hiint(cabs1(x[0])) & 0x7fffffff : -1;
#pragma unroll
      for (int q = 0; q < 7; ++q) pb[q] = c.row[q + 9];
      rc = recip_pivot(x[0]);
      best = wave_max_int(key);
#pragma unroll
      for (int q = 1; q < 8; ++q) x[q] = fmsc(x[q + 1], m, mkc(pa[q].x, pa[q].y));
#pragma unroll
      for (int q = 8; q < NB - 1; ++q) x[q] = fmsc(x[q + 1], m, mkc(pb[q - 8].x, pb[q - 8].y));
      x[NB - 1] = -m;
    }
    for (int jj = nb; jj < NB; ++jj) {  // the last panel: rotate on
      const cd t = x[0];
#pragma unroll
      for (int q = 1; q < NB; ++q) x[q - 1] = x[q];
      x[NB - 1] = t;
    }
    if (row < n) {
#pragma unroll
      for (int c = 0; c < NB; ++c)
        if (c < nb) a[(unsigned)(row * lda + k0 + c)] = x[c];
    }
    __syncthreads();  // G and ord of this panel are read by the other wavefronts
  }
  if (row < n) {
    const int k = ord[row];
    if (k >= c0 && k < c1) perm[item * n + k] = row;
  }
  if (tid == 0 && info && (c0 == 0 || (first_zero && info[item] == 0))) info[item] = first_zero;
}

// ------------------------------------------------------------ right-hand sides
// Panels j0 .. j1 - 1 on the strips of B (n x m).  LAST: the rows come out in the
// order of the unknowns (after the last panel); else they stay where they are.
template <int RB, int CB, bool LAST>
__global__ __launch_bounds__(512) void gj_strips_kernel(int n, int m, int j0, int j1, const cd* A, int lda,
                                                        long long sA, cd* B, int ldb, long long sB,
                                                        const int* __restrict__ perm, int strips, int xcd_remap) {
  extern __shared__ lcd sm[];
  constexpr int YC = 16 * CB + 1;
  lcd* Y = sm;                                               // 2 x 17 x YC
  int* ord = reinterpret_cast<int*>(Y + 2 * (NB + 1) * YC);  // 16 RB nw
  unsigned bid = blockIdx.x;
  if (xcd_remap) {  // gridDim.x % 8 == 0: the strips of one system on one XCD
    const unsigned per = gridDim.x / 8;
    bid = (bid % 8) * per + bid / 8;
  }
  const long long item = bid / strips;
  const int col0 = (int)(bid % strips) * 16 * CB;
  const cd* a = A + item * sA;
  cd* b = B + item * sB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int row0 = wave * 16 * RB;
  const int rows = (blockDim.x >> 6) * 16 * RB;
  const int k0 = j0 * NB, k1 = min(n, j1 * NB);
  for (int k = tid; k < rows; k += blockDim.x) ord[k] = 1 << 30;
  __syncthreads();
  for (int k = k0 + tid; k < k1; k += blockDim.x) ord[perm[item * n + k]] = k;
  Strip<RB, CB> x;
#pragma unroll
  for (int t = 0; t < RB; ++t)
#pragma unroll
    for (int u = 0; u < CB; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gr = row0 + t * 16 + lk + 4 * r, gc = col0 + u * 16 + li;
        const cd v = b[(long long)min(gr, n - 1) * ldb + min(gc, m - 1)];  // (past the edges: never stored)
        x.re[t][u][r] = v.x;
        x.im[t][u][r] = v.y;
      }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < RB; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) x.slot[t][r] = ord[row0 + t * 16 + lk + 4 * r];
  apply_panels(x, a, lda, n, j0, j1, k1 - (j1 - 1) * NB, Y, row0, li, lk);
#pragma unroll
  for (int t = 0; t < RB; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gr = row0 + t * 16 + lk + 4 * r;
      if (gr >= n) continue;
      const int k = LAST ? x.slot[t][r] : gr;
#pragma unroll
      for (int u = 0; u < CB; ++u) {
        const int gc = col0 + u * 16 + li;
        if (gc < m) b[(long long)k * ldb + gc] = mkc(x.re[t][u][r], x.im[t][u][r]);
      }
    }
}

template <int RB, int CB, bool LAST>
int launch_strips(hipStream_t s, int n, int m, int j0, int j1, Mat A, Mat B, int batch, const int* perm) {
  const int th = 64 * ((n + 16 * RB - 1) / (16 * RB));
  const int strips = (m + 16 * CB - 1) / (16 * CB);
  const long long blocks = (long long)strips * batch;
  KHX_REQUIRE(blocks < (1ll << 31), "zgesv: grid too large");
  const size_t lds = (size_t)2 * (NB + 1) * (16 * CB + 1) * sizeof(lcd) + (size_t)(th / 64) * 16 * RB * sizeof(int);
  gj_strips_kernel<RB, CB, LAST><<<dim3((unsigned)blocks), dim3(th), lds, s>>>(
      n, m, j0, j1, A.p, A.ld, A.stride, B.p, B.ld, B.stride, perm, strips, blocks % 8 == 0 ? 1 : 0);
  KHX_LAUNCH_CHECK();
  return 0;
}

// Rows per wavefront: as few as give four wavefronts.  Strips of 32 columns halve
// the traffic of G (n = 338, 512 systems: 3.4 against 3.8 ms); narrower ones
// spread a small batch over more CUs.
template <bool LAST>
int strips_sized(hipStream_t s, int n, int m, int j0, int j1, Mat A, Mat B, int batch, const int* perm) {
  const int rb = n <= 64 ? 1 : n <= 128 ? 2 : n <= 192 ? 3 : n <= 256 ? 4 : n <= 384 ? 3 : 4;
  const int nw = (n + 16 * rb - 1) / (16 * rb);
  const bool wide = m > 16 && (long long)batch * ((m + 31) / 32) * nw >= 2048;
  switch (rb * 2 + (wide ? 1 : 0)) {
    case 2: return launch_strips<1, 1, LAST>(s, n, m, j0, j1, A, B, batch, perm);
    case 3: return launch_strips<1, 2, LAST>(s, n, m, j0, j1, A, B, batch, perm);
    case 4: return launch_strips<2, 1, LAST>(s, n, m, j0, j1, A, B, batch, perm);
    case 5: return launch_strips<2, 2, LAST>(s, n, m, j0, j1, A, B, batch, perm);
    case 6: return launch_strips<3, 1, LAST>(s, n, m, j0, j1, A, B, batch, perm);
    case 7: return launch_strips<3, 2, LAST>(s, n, m, j0, j1, A, B, batch, perm);
    case 8: return launch_strips<4, 1, LAST>(s, n, m, j0, j1, A, B, batch, perm);
    default: return launch_strips<4, 2, LAST>(s, n, m, j0, j1, A, B, batch, perm);
  }
}

template <int RB>
int launch_factor(hipStream_t s, int n, int c0, int c1, Mat A, int batch, int* perm, int* info) {
  const int nw = (n + 16 * RB - 1) / (16 * RB);
  const size_t lds = (size_t)(nw * 16 + 2 * (NB + 1)) * YS * sizeof(lcd) + 2 * GJ_MAX_WAVES * (sizeof(Candidate) + sizeof(int2)) +
                     (size_t)nw * 16 * RB * sizeof(int);
  KHX_TRY(ensure_dynamic_lds((const void*)gj_factor_kernel<RB>, lds));
  gj_factor_kernel<RB><<<dim3((unsigned)batch), dim3(64 * nw), lds, s>>>(n, c0, c1, A.p, A.ld, A.stride, perm, info);
  KHX_LAUNCH_CHECK();
  return 0;
}

}  // namespace

constexpr int GJ_MAX_N = 512;

bool zgj_fits(int n, int m) { return n >= 1 && n <= GJ_MAX_N && m >= 1; }

// A X = B: A (n x n) destroyed, B (n x m) overwritten by X, perm: n ints per
// item of scratch; info[b] = first zero pivot (1-based) or 0.
int zgj_solve(hipStream_t s, int n, int m, Mat A, Mat B, int batch, int* perm, int* info) {
  if (batch <= 0 || n <= 0) return 0;
  KHX_REQUIRE(zgj_fits(n, m), "zgj_solve: order out of range");
  KHX_REQUIRE((A.stride != 0 && B.stride != 0) || batch == 1, "zgesv: operands cannot be broadcast");
  KHX_REQUIRE((long long)A.ld * n < (1ll << 31), "zgesv: row stride too large");
  ProfScope ps("zgesv_kernel", s);
  // Columns factored by one launch before the others are brought up to date.  One
  // workgroup per system factors, so few systems leave most of the chip to the
  // updates' strips, and panels of a launch that reads back little cost little:
  // 64 columns below 256 systems (n = 338, 16 systems: 1.01 ms against 1.14 with
  // 128 and 1.82 in one launch; n = 162, 64: 0.37 / 0.38 / 0.40).  Beyond, the CUs
  // are full either way: 128 columns where G outgrows what a CU's cache keeps
  // (n = 338, 512 systems: 7.4 / 7.1 / 7.5 ms), all at once up to n = 192 (n =
  // 162, 1 024: 2.06 / 1.99 / 1.90).
  const int wb = batch < 256 ? 64 : n > 192 ? 128 : n;
  // Rows per wavefront of the factorization: 64 while one or two wavefronts hold
  // the matrix (fewer barriers per pivot; n = 98, 1 000 systems: 0.56 ms against
  // 0.72 with 48), 48 where 64 would leave three wavefronts on four SIMDs (n =
  // 162, 2 048: 3.7 against 4.0 ms), 64 again where four or more are needed
  // (n = 338, 48: 1.48 against 1.53 ms).
  const int rbf = n > 128 && n <= 192 ? 3 : 4;
  for (int c0 = 0; c0 < n; c0 += wb) {
    const int c1 = c0 + wb < n ? c0 + wb : n;
    if (rbf == 3)
      KHX_TRY(launch_factor<3>(s, n, c0, c1, A, batch, perm, info));
    else
      KHX_TRY(launch_factor<4>(s, n, c0, c1, A, batch, perm, info));
    if (c1 < n)
      KHX_TRY(strips_sized<false>(s, n, n - c1, c0 / NB, c1 / NB, A, Mat{A.p + c1, A.ld, A.stride}, batch, perm));
  }
  return strips_sized<true>(s, n, m, 0, (n + NB - 1) / NB, A, B, batch, perm);
}

}  // namespace khx
