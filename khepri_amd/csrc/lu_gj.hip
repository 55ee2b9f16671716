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
// gj_factor_kernel: 32 columns and more in one launch, one workgroup per system.  A
//   panel's columns are loaded into MFMA accumulators, the launch's earlier
//   panels are applied to them (left-looking: A is read and written once), and
//   the panel is eliminated where it lies, a column per lane of 16 and 16 rows per
//   four registers.  A pivot step: the rows' keys are made as the values are, the
//   wavefronts' candidate rows go through LDS as one 16-byte word per lane, the
//   multipliers come from the column's lane by DPP; one barrier.  (One row per lane
//   costs 33 LDS words per step and wavefront instead of 3, at 30 to 36 clocks
//   each: n = 50, 302 systems 0.105 -> 0.087 ms, n = 338, 2 systems 0.88 -> 0.72.)
// gj_strips_kernel: one workgroup per system and strip of 16 CB columns, of B or
//   of the columns of A still to be factored.  The strip stays in MFMA
//   accumulators from its load to its store while the panels pass by: 8 n^2
//   operations per column on the matrix cores with B moved once; the 16 pivot
//   rows of a panel go through LDS, G comes from L2 (the strips of one system run
//   on one XCD).
// The multi-launch LU (lu_blocked.hip) needs 11 panel launches, as many trailing
// updates and 22 leaf launches for n = 162 and moves the trailing matrix once per
// panel.  Measured, LU -> here, ms: n = 50 (50 right-hand sides) 2 systems 0.28 ->
// 0.055, 4 096 systems 4.4 -> 0.37; n = 162 (162) 2 048 systems 7.0 -> 3.55; n =
// 338 (338) 512 systems 11.1 -> 6.8, 2 systems 0.72.  The strips keep the FP64
// matrix pipe 67 % busy (n = 162, 2 048 systems), the factorization 31 %: it is
// bound by the latency of its pivot steps (0.6 to 0.9 us: the updates and keys of 16
// registers 0.25, candidates, barrier and winner 0.2, reciprocal 0.1) and of a
// panel's loads and products.
// Error: forward error as an LU's; the residual of an ill-conditioned system can
// be larger (Gauss-Jordan is not row-wise backward stable).  Most systems it serves
// are well conditioned (the slice and the doublings, formed against a medium in
// which a lossless S-matrix is unitary); the last step to the gap and the junctions
// of a chain are not near a pole of a layer's S-matrix against the gap.  There R
// and T come out as with an LU: 155 stacks of order 10 to 30 placed on such poles
// (cond(D) up to 1e7) against 80-bit arithmetic, the worst propagating amplitude's
// error as the mean of its logarithm and the largest: here 3.6e-13 and 9.0e-9, the
// same with LU 3.1e-13 and 9.3e-9, through the modes with LU 3.4e-13 and 1.2e-8 (the
// rounding of the layer's input is most of it); 0.001 of frequency beside them
// 1.9e-14 and 5.6e-13, 1.9e-14 and 6.0e-13, 2.5e-14 and 6.8e-13.
#include "khx_internal.h"
#include "khx_prof.h"

namespace khx {

namespace {

typedef double gj_d4 __attribute__((ext_vector_type(4)));
constexpr int NB = 16;      // panel width
constexpr int YS = NB + 1;  // LDS row stride

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
constexpr int GJ_MAX_WAVES = 8;
constexpr int ROW_BITS = 9;                                    // rows < GJ_MAX_N
constexpr int KEY_MASK = 0x7fffffff & ~((1 << ROW_BITS) - 1);  // a key's magnitude bits
constexpr int CLOSED = (int)0x80000000;

// lane JJ of every 16 lanes to all of them
template <int JJ>
__device__ __forceinline__ double bcast16(double v) {
  return __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(v), 0x150 + JJ, 0xf, 0xf, true));
}

// every lane's value to the lane four down, around the 16
__device__ __forceinline__ double rotate4(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x12c, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x12c, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// The panel under elimination, where the matrix cores left it: entry i = 4 t + r
// of lane l is row 16 t + l / 16 + 4 r of the wavefront, column l % 16.  Vectors,
// so that a row found at run time is one indexed register move.
template <int RB>
struct PanelRegs {
  typedef double vec __attribute__((ext_vector_type(RB == 3 ? 16 : 4 * RB)));
  typedef int ivec __attribute__((ext_vector_type(RB == 3 ? 16 : 4 * RB)));
  vec re, im;
  // row number, with the sign bit set once the row has been a pivot (or is none)
  ivec tag;
};

// A row's key for being the pivot of this lane's column: the high bits of |re| +
// |im| (to 2^-11), then the row number.
__device__ __forceinline__ int pivot_key(double re, double im, int tag) {
  return (__double2hiint(fabs(re) + fabs(im)) & KEY_MASK) | tag;
}

// the maximum of column JJ's lanes
template <int JJ>
__device__ __forceinline__ int column_max(int key) {
  const int a = max(__builtin_amdgcn_readlane(key, JJ), __builtin_amdgcn_readlane(key, 16 + JJ));
  const int b = max(__builtin_amdgcn_readlane(key, 32 + JJ), __builtin_amdgcn_readlane(key, 48 + JJ));
  return max(a, b);
}

struct FactorLds {
  lcd* cand;  // 2 x GJ_MAX_WAVES rows of 16 and a spare one
  int* keys;  // 2 x GJ_MAX_WAVES
};

// Column k, which lanes JJ of each 16 hold.  best: the wavefront's key for it, then
// for the next column's; sc: what this lane's column is multiplied with at the
// end of the panel; pivot: the row this lane's column was eliminated with.
template <int RB, int JJ>
__device__ __forceinline__ void eliminate(PanelRegs<RB>& x, int& best, cd& sc, int& pivot, int& first_zero, int k,
                                          const FactorLds& sm, int nw, int wave, int row0, int li, int lk) {
  constexpr int buf = (JJ & 1) * GJ_MAX_WAVES;
  {
    const int at = (best & ((1 << ROW_BITS) - 1)) - row0;
    const int i = at >> 2;
    // (the other rows' lanes write to a spare row, and all lanes the key: no branches)
    sm.cand[(lk == (at & 3) ? buf + wave : 2 * GJ_MAX_WAVES) * 16 + li] = lcd{x.re[i], x.im[i]};
    sm.keys[buf + wave] = best;
  }
  __syncthreads();
  int kbest = best;
  if (nw > 1) {
    const int4 a = *reinterpret_cast<const int4*>(sm.keys + buf), b = *reinterpret_cast<const int4*>(sm.keys + buf + 4);
    kbest = __builtin_amdgcn_readfirstlane(max(max(max(a.x, a.y), max(a.z, a.w)), max(max(b.x, b.y), max(b.z, b.w))));
  }
  const int prow = kbest & ((1 << ROW_BITS) - 1);
  const int w = prow / (16 * RB);
  const lcd pl = sm.cand[(buf + w) * 16 + li];
  const cd p = mkc(pl.x, pl.y);
  if ((kbest & KEY_MASK) == 0 && first_zero == 0) first_zero = k + 1;
  const cd mine = recip_pivot(p);
  const cd rc = mkc(bcast16<JJ>(mine.x), bcast16<JJ>(mine.y));
  cd y = p * rc;
  const bool own = li == JJ;
  y.x = own ? 0.0 : y.x;  // the column itself stays, until it is scaled with sc
  y.y = own ? 0.0 : y.y;
  sc.x = own ? -rc.x : sc.x;
  sc.y = own ? -rc.y : sc.y;
  pivot = own ? prow : pivot;
  // (no branch on whether the row is this wavefront's: the registers would be
  // copied where its two sides join)
  const int at = w == wave ? prow - row0 : 0, ip = at >> 2;
  const bool hit = w == wave && lk == (at & 3);
  const int tp = x.tag[ip];
  x.tag[ip] = hit ? CLOSED | prow : tp;
  int key = CLOSED;
#pragma unroll
  for (int i = 0; i < 4 * RB; ++i) {
    const double mr = bcast16<JJ>(x.re[i]), mi = bcast16<JJ>(x.im[i]);
    x.re[i] = fma(mi, y.y, fma(-mr, y.x, x.re[i]));
    x.im[i] = fma(-mi, y.x, fma(-mr, y.y, x.im[i]));
    const int c = pivot_key(x.re[i], x.im[i], x.tag[i]);
    key = i == 0 ? c : max(key, c);
  }
  const double pr = x.re[ip], pi = x.im[ip];  // the pivot row
  x.re[ip] = hit ? (own ? -1.0 : y.x) : pr;
  x.im[ip] = hit ? y.y : pi;
  best = column_max<JJ + 1>(key);
}

// Columns c0 .. c1 - 1 (c0 a multiple of 16), to which the panels before c0 have
// been applied.  Workgroups of ceil(n / (16 RB)) wavefronts.
template <int RB>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(RB <= 3 ? 3 : 2))) void gj_factor_kernel(
    int n, int c0, int c1, cd* A, int lda, long long sA, int* perm, int* info) {
  extern __shared__ lcd sm[];
  const int nw = blockDim.x >> 6;
  lcd* Y = sm;  // 2 x 17 x YS
  FactorLds fl;
  fl.cand = Y + 2 * (NB + 1) * YS;
  fl.keys = reinterpret_cast<int*>(fl.cand + (2 * GJ_MAX_WAVES + 1) * 16);
  int* ord = fl.keys + 2 * GJ_MAX_WAVES;  // 16 RB nw
  const long long item = blockIdx.x;
  cd* a = A + item * sA;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int row0 = wave * 16 * RB;
  int first_zero = 0;
  for (int e = tid; e < 16 * RB * nw; e += blockDim.x) ord[e] = 1 << 30;
  if (tid < 2 * GJ_MAX_WAVES) fl.keys[tid] = CLOSED;
  __syncthreads();
  for (int k = tid; k < c0; k += blockDim.x) ord[perm[item * n + k]] = k;
  __syncthreads();
  for (int k0 = c0; k0 < c1; k0 += NB) {
    const int nb = min(NB, n - k0);
    PanelRegs<RB> x;
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
          x.tag[4 * t + r] = gr | (gr < n && st.slot[t][r] == 1 << 30 ? 0 : CLOSED);
        }
      apply_panels(st, a, lda, n, c0 / NB, k0 / NB, NB, Y, row0, li, lk);
#pragma unroll
      for (int t = 0; t < RB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x.re[4 * t + r] = st.re[t][0][r];
          x.im[4 * t + r] = st.im[t][0][r];
        }
    }
    int key = 0;
#pragma unroll
    for (int i = 0; i < 4 * RB; ++i) {
      const int c = pivot_key(x.re[i], x.im[i], x.tag[i]);
      key = i == 0 ? c : max(key, c);
    }
    cd sc = mkc(0.0, 0.0);
    int best = column_max<0>(key), col = li, pivot = 0;
    // Four columns per pass through the code, then the columns move four lanes
    // down: which lane is read is part of the instruction, and sixteen copies of
    // the step (50 KB) would be fetched more slowly than they run.
#pragma unroll 1
    for (int j = 0; j < nb; j += 4) {
      eliminate<RB, 0>(x, best, sc, pivot, first_zero, k0 + j, fl, nw, wave, row0, li, lk);
      if (j + 1 < nb) eliminate<RB, 1>(x, best, sc, pivot, first_zero, k0 + j + 1, fl, nw, wave, row0, li, lk);
      if (j + 2 < nb) eliminate<RB, 2>(x, best, sc, pivot, first_zero, k0 + j + 2, fl, nw, wave, row0, li, lk);
      if (j + 3 < nb) eliminate<RB, 3>(x, best, sc, pivot, first_zero, k0 + j + 3, fl, nw, wave, row0, li, lk);
#pragma unroll
      for (int i = 0; i < 4 * RB; ++i) {
        x.re[i] = rotate4(x.re[i]);
        x.im[i] = rotate4(x.im[i]);
      }
      sc = mkc(rotate4(sc.x), rotate4(sc.y));
      pivot = __builtin_amdgcn_mov_dpp(pivot, 0x12c, 0xf, 0xf, true);
      col = (col + 4) & 15;
    }
    if (wave + lk == 0 && col < nb) ord[pivot] = k0 + col;
#pragma unroll
    for (int i = 0; i < 4 * RB; ++i) {
      const int gr = row0 + 4 * i + lk;
      if (gr < n && col < nb) a[(unsigned)(gr * lda + k0 + col)] = mkc(x.re[i], x.im[i]) * sc;
    }
    __syncthreads();  // G and ord of this panel are read by the other wavefronts
  }
  for (int row = tid; row < n; row += blockDim.x) {
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
  const size_t lds = ((size_t)2 * (NB + 1) * YS + (2 * GJ_MAX_WAVES + 1) * 16) * sizeof(lcd) +
                     ((size_t)2 * GJ_MAX_WAVES + nw * 16 * RB) * sizeof(int);
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
  // updates' strips: 32 columns up to 32 systems (from n = 129; n = 338, 2 systems:
  // 0.72 ms against 0.77 with 64 and 1.6 in one launch), 64 below 256 (n = 338, 64:
  // 1.45 / 1.49 / 1.52 ms with 64 / 32 / 128; n = 162, 64: 0.30 / 0.31 / 0.32).
  // Beyond, the CUs are full either way: 128 columns where G outgrows what a CU's
  // cache keeps (n = 338, 512 systems: 7.1 / 6.8 / 7.2 ms with 64 / 128 / all), all
  // at once up to n = 192 (n = 162, 1 024: 1.94 / 1.90 / 1.87).
  const int wb = batch <= 32 && n > 128 ? 32 : batch < 256 ? 64 : n > 192 ? 128 : n;
  // Rows per wavefront of the factorization, 16 rb.  A step's updates go with rb,
  // the rest of it with the wavefronts: four wavefronts on the four SIMDs while a
  // CU has one or two systems (n = 50, 128 systems: 0.061 ms against 0.076 in one
  // wavefront; n = 98, 128: 0.154 / 0.17), as few as hold the matrix beyond (n =
  // 50, 2 048: 0.25 / 0.20; n = 98, 1 000: 0.55 / 0.53).  n = 162 in four
  // wavefronts of 48 rows when the CUs are full (512 systems: 0.94 against 0.98).
  const bool full = batch > 512;
  const int rbf = n <= 64 ? (full ? 4 : 1) : n <= 128 ? (full ? 4 : 2) : n <= 192 && batch >= 256 ? 3 : 4;
  for (int c0 = 0; c0 < n; c0 += wb) {
    const int c1 = c0 + wb < n ? c0 + wb : n;
    switch (rbf) {
      case 1: KHX_TRY(launch_factor<1>(s, n, c0, c1, A, batch, perm, info)); break;
      case 2: KHX_TRY(launch_factor<2>(s, n, c0, c1, A, batch, perm, info)); break;
      case 3: KHX_TRY(launch_factor<3>(s, n, c0, c1, A, batch, perm, info)); break;
      default: KHX_TRY(launch_factor<4>(s, n, c0, c1, A, batch, perm, info));
    }
    if (c1 < n)
      KHX_TRY(strips_sized<false>(s, n, n - c1, c0 / NB, c1 / NB, A, Mat{A.p + c1, A.ld, A.stride}, batch, perm));
  }
  return strips_sized<true>(s, n, m, 0, (n + NB - 1) / NB, A, B, batch, perm);
}

}  // namespace khx
