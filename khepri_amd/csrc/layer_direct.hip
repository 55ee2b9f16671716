// S-matrix of a patterned layer without its modes.
//
// The layer's fields obey E' = P H, H' = Q E (z in units of 1/k0), so its
// S-matrix is a function of F = P Q alone: with x = (k0 d / 2) sqrt(F) the even
// and odd excitations of the symmetric slab see the face relations
//   even: E = cosh(x) e,  H = -(k0 d / 2) Q [sinh(x)/x] e
//   odd:  E = -(k0 d / 2) [sinh(x)/x] P h,  H = cosh(x) h,
// entire functions of F that need no eigenvectors (the reference goes through
// eig(P Q), khepri/alternative.py:158-195; the S-matrix it forms is this one).
// The slab is cut into 2^s equal slices so that |x| <= LAYER_THETA, and
//   1. cosh and sinh(x)/x of the slice come, up to one common factor that
//      cancels, from the diagonal Pade approximant [17/17] of e^{2x}: its even
//      and odd parts are polynomials of degree 8 in F: F^2, [F^3 | F^4] and one
//      n x 2n product for both polynomials;
//   2. the slice's even and odd reflections are formed against a reference
//      medium in which every harmonic carries power, H = -Vr E with
//      Vr = -i [[0, 1], [-1, 0]] (the gap's normal-incidence admittance).  For a
//      lossless layer that S-matrix is unitary, so nothing below is
//      ill-conditioned: the gap's own evanescent orders would give poles at
//      slice thicknesses that carry a guided mode;
//   3. s doublings, E/O = S12 (1 -/+ S11)^-1 S12, S11' = S11 + (E - O)/2,
//      S12' = (E + O)/2;
//   4. the change to the gap medium.  Its reflection seen from the reference
//      medium is, per harmonic, R1 = [[kx^2 - ky^2, 2 kx ky], [2 kx ky,
//      ky^2 - kx^2]] / (1 + kz)^2, and for either parity
//      G' = R1 + (1 - R1) (1 + G R1)^-1 G (1 + R1).
// Work: 48 n^3 + 21 n^3 (slice) + 37 n^3 per doubling + 21 n^3 real operations,
// all products and solves of full matrices, against a non-symmetric
// eigenproblem whose bulge chase leaves the matrix cores idle.  Measured
// through the eigensolver -> here: 24 layers of n = 338 179 -> 8.5 ms; 4 096
// disc stacks of n = 162 424 -> 103 ms; the error against 64-bit references is
// the same or smaller (n = 50 against 80-bit arithmetic: 1e-14..1e-13 -> 2e-15..
// 4e-14) while the outermost harmonic is within |K| = 25.  For longer waves the
// change to the gap medium costs the entries between evanescent orders more than the
// modes do (|K| = 100: 1e-12 -> 5e-12, |K| = 400: 3e-11 -> 2e-10 of the largest
// entry); those between propagating orders stay 10 to 100 times nearer.
#include "khx_internal.h"

namespace khx {

namespace {

__device__ __forceinline__ cd kz_gap(cd x, cd y) {  // khepri/alternative.py:92-96
  const cd kz2 = mkc(1.0, 0.0) - x * x - y * y;
  if (kz2.x < 0.0) {
    const cd r = sqrtc(-kz2);
    return mkc(r.y, -r.x);
  }
  return sqrtc(kz2);
}

// Coefficients of the even and odd part of the [17/17] numerator of e^{2x}
// (even part: sum c_j F^j, odd part / x: sum s_j F^j, F = x^2), over c_0.  The
// degree: [13/13] holds to |x| = 2.75 with 8 n^3 less work, [17/17] to 4.4 on both
// axes; half a doubling of 37 n^3 is saved on average, and cosh(4) = 27 still
// leaves the slice as accurate as the modes (cosh(5.5) = 120, [21/21], does not).
struct PadeCoef {
  double c[9], s[9];
};
constexpr int PADE_M = 17;
constexpr PadeCoef pade_coef() {
  PadeCoef p{};
  // numerator of e^y: b_j = (2m - j)! m! / ((2m)! j! (m - j)!), y = 2x
  double b = 1.0, pow2 = 1.0;
  for (int j = 0; j <= PADE_M; ++j) {
    if (j % 2 == 0)
      p.c[j / 2] = b * pow2;
    else
      p.s[j / 2] = b * pow2;
    b = b * (PADE_M - j) / ((2 * PADE_M - j) * (j + 1.0));
    pow2 *= 2.0;
  }
  return p;
}
__constant__ const PadeCoef PADE = pade_coef();

dim3 grid_ew(long long total) {
  long long g = (total + 255) / 256;
  if (g > 131072) g = 131072;
  if (g < 1) g = 1;
  return dim3((unsigned)g);
}

// ------------------------------------------------------------ |x| of a layer
// Largest |eigenvalue| of F by power iteration, one workgroup per item, the
// vector in LDS.  F v = J Q v + K C^-1 K^T (C v) needs three N x N matrix-vector
// products and never forms F.  Sixteen lanes take a row, summed by DPP: a product
// is one pass for N <= 32 and waits for one reduction of four steps (a wavefront
// per row waited for six shuffles at every eighth row: a call with 1 item of N =
// 25 83 -> 38 us, with 1 024 of N = 81 737 -> 175).
// One step's growth |F v| / |v| approaches the largest |eigenvalue| from below
// where F is close to normal (its largest modes crowd near |K|^2 of the outermost
// harmonics, where the start vector is concentrated).  Where the permittivity
// changes sign they come in pairs of nearly opposite sign, and one step grows as
// much as the next shrinks: the estimate is the largest of the last step's growth
// and the geometric means over the last 2 to LAYER_POWER_MEANS steps.  Against
// eigenvalues from numpy, 20 000 drawn maps: at least 0.87 of the true |x| (0.89
// without sign changes and metals; the last step alone: 0.50), up to 2.3 times it
// where the sign changes, 1.04 elsewhere.  So a slice has |x| <= 4 / 0.87 = 4.6,
// where the approximant's error is 6e-17 (1e-16 at 4.7, 1e-15 at 5, 4e-13 at 6).
constexpr int LAYER_POWER_STEPS = 8;
constexpr int LAYER_POWER_MEANS = 6;
constexpr int SCALE_THREADS = 512;

// the sum over 16 lanes, in all of them
__device__ __forceinline__ double row_sum16(double v) {
#define KHX_ROR(n)                                                                            \
  v += __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + n, 0xf, 0xf, true), \
                        __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + n, 0xf, 0xf, true));
  KHX_ROR(8)
  KHX_ROR(4)
  KHX_ROR(2)
  KHX_ROR(1)
#undef KHX_ROR
  return v;
}

__global__ __launch_bounds__(SCALE_THREADS) void layer_scale_kernel(
    const cd* __restrict__ C, const cd* __restrict__ IC, long long cstride, const cd* __restrict__ kx,
    const cd* __restrict__ ky, int N, const double* __restrict__ k0d, double* __restrict__ est) {
  extern __shared__ cd sm[];
  cd* v = sm;           // 2N
  cd* w = sm + 2 * N;   // 2N: C v1, C v2
  cd* u = sm + 4 * N;   // N
  cd* fx = sm + 5 * N;  // kx
  cd* fy = sm + 6 * N;  // ky
  __shared__ double red[SCALE_THREADS / 64], growth[LAYER_POWER_STEPS];  // growth: thread 0's
  const long long b = blockIdx.x;
  const cd* c = C + b * cstride;
  const cd* ic = IC + b * cstride;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, li = tid & 15;
  constexpr int NW = SCALE_THREADS / 64;
  for (int h = tid; h < N; h += SCALE_THREADS) {
    const cd x = kx[b * N + h], y = ky[b * N + h];
    fx[h] = x;
    fy[h] = y;
    const double k2 = 1.0 + abs2c(x) + abs2c(y);
    // fixed signs that no symmetry of the harmonics repeats
    v[h] = mkc(k2 * ((h * 7 + 3) % 11 - 4.7), k2 * ((h * 5 + 1) % 7 - 2.6));
    v[N + h] = mkc(k2 * ((h * 3 + 2) % 13 - 5.1), k2 * ((h * 11 + 4) % 9 - 4.3));
  }
  __syncthreads();
  auto norm2 = [&](const cd* p) {
    double s = 0.0;
    for (int h = tid; h < 2 * N; h += SCALE_THREADS) s += abs2c(p[h]);
    s = wave_sum(s);
    if (lane == 0) red[wid] = s;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < NW; ++q) t += red[q];
    __syncthreads();
    return t;
  };
  double n0 = norm2(v);
  for (int it = 0; it < LAYER_POWER_STEPS; ++it) {
    const double sc = 1.0 / sqrt(n0);
    for (int r = tid >> 4; r < N; r += SCALE_THREADS / 16) {
      cd a1 = mkc(0.0, 0.0), a2 = mkc(0.0, 0.0);
      for (int j = li; j < N; j += 16) {
        const cd m = c[(long long)r * N + j];
        a1 = fmac(a1, m, v[j]);
        a2 = fmac(a2, m, v[N + j]);
      }
      a1 = mkc(row_sum16(a1.x), row_sum16(a1.y));
      a2 = mkc(row_sum16(a2.x), row_sum16(a2.y));
      if (li == 0) {
        w[r] = a1;
        w[N + r] = a2;
        u[r] = fx[r] * a1 + fy[r] * a2;
      }
    }
    __syncthreads();
    for (int r = tid >> 4; r < N; r += SCALE_THREADS / 16) {
      cd a = mkc(0.0, 0.0);
      for (int j = li; j < N; j += 16) a = fmac(a, ic[(long long)r * N + j], u[j]);
      a = mkc(row_sum16(a.x), row_sum16(a.y));
      if (li == 0) {
        const cd x = fx[r], y = fy[r], t = y * v[r] - x * v[N + r];
        w[r] = sc * (x * a + y * t - w[r]);
        w[N + r] = sc * (y * a - x * t - w[N + r]);
      }
    }
    __syncthreads();
    for (int h = tid; h < 2 * N; h += SCALE_THREADS) v[h] = w[h];
    __syncthreads();
    n0 = norm2(v);  // = |F v|^2 / |v|^2 of this step
    if (tid == 0) growth[it] = n0;
  }
  if (tid == 0) {
    bool shrank = false;  // no mean exceeds the last step otherwise
#pragma unroll
    for (int w = 2; w <= LAYER_POWER_MEANS; ++w) shrank |= growth[LAYER_POWER_STEPS - w] > n0;
    double best = n0;
    if (shrank) {
      double sum = log2(n0);
      for (int w = 2; w <= LAYER_POWER_MEANS; ++w) {
        sum += log2(growth[LAYER_POWER_STEPS - w]);
        const double mean = exp2(sum / w);
        if (mean > best) best = mean;
      }
    }
    est[b] = 0.5 * fabs(k0d[b]) * sqrt(sqrt(best));
  }
}

// ------------------------------------------------------------ F
// T = [Kx C | Ky C] (N x 2N)
__global__ void scale_rows_kernel(const cd* __restrict__ C, long long cstride, const cd* __restrict__ kx,
                                  const cd* __restrict__ ky, int N, int batch, cd* __restrict__ T) {
  const long long per = (long long)N * N, total = per * batch;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const long long b = e / per;
    const int rc = (int)(e % per), r = rc / N, c = rc % N;
    const cd v = C[b * cstride + rc];
    cd* t = T + b * 2 * per + (long long)r * 2 * N;
    t[c] = kx[b * N + r] * v;
    t[N + c] = ky[b * N + r] * v;
  }
}

// tau^2 F into the first n columns of the (n x 4n) power buffer:
//   F = [Kx; Ky] (C^-1 [Kx C | Ky C]) + J Q,
//   J Q = [[Ky^2 - C, -Kx Ky], [-Kx Ky, Kx^2 - C]],  G = C^-1 [Kx C | Ky C]
// A non-finite entry marks the item (the reference's eig raises on it).
__global__ void build_f_kernel(const cd* __restrict__ G, const cd* __restrict__ C, long long cstride,
                               const cd* __restrict__ kx, const cd* __restrict__ ky, const double* __restrict__ k0d,
                               double scale, int N, int batch, cd* __restrict__ W4, int* __restrict__ bad) {
  const int n = 2 * N;
  const long long per = (long long)N * N, total = per * batch;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const long long b = e / per;
    const int rc = (int)(e % per), r = rc / N, c = rc % N;
    const double tau = 0.5 * k0d[b] * scale, t2 = tau * tau;
    const cd x = kx[b * N + r], y = ky[b * N + r];
    const cd g1 = G[b * 2 * per + (long long)r * 2 * N + c], g2 = G[b * 2 * per + (long long)r * 2 * N + N + c];
    const cd cc = C[b * cstride + rc];
    cd tl = x * g1 - cc, tr = x * g2, bl = y * g1, br = y * g2 - cc;
    if (r == c) {
      tl = tl + y * y;
      tr = tr - x * y;
      bl = bl - x * y;
      br = br + x * x;
    }
    const double probe = (tl.x + tl.y) + (tr.x + tr.y) + (bl.x + bl.y) + (br.x + br.y);
    if (!isfinite(probe) || !isfinite(t2)) bad[b] = 1;
    cd* w = W4 + b * 16 * per;  // n * 4n = 16 N^2
    w[(long long)r * 4 * n + c] = t2 * tl;
    w[(long long)r * 4 * n + N + c] = t2 * tr;
    w[(long long)(N + r) * 4 * n + c] = t2 * bl;
    w[(long long)(N + r) * 4 * n + N + c] = t2 * br;
  }
}

// Both polynomials split at F^4: U = [c5 F + c6 F^2 + c7 F^3 + c8 F^4 | s5 F + ...]
// and CS = [c0 + c1 F + ... + c4 F^4 | s0 + ...]; then CS += F^4 U.
__global__ void pade_parts_kernel(const cd* __restrict__ W4, int n, int batch, cd* __restrict__ U,
                                  cd* __restrict__ CS) {
  const long long per = (long long)n * n, total = per * batch;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const long long b = e / per;
    const int rc = (int)(e % per), r = rc / n, c = rc % n;
    const cd* w = W4 + b * 4 * per + (long long)r * 4 * n + c;
    const cd f1 = w[0], f2 = w[n], f3 = w[2 * n], f4 = w[3 * n];
    const cd d = mkc(r == c ? 1.0 : 0.0, 0.0);
    const long long o = b * 2 * per + (long long)r * 2 * n + c;
    U[o] = PADE.c[5] * f1 + PADE.c[6] * f2 + PADE.c[7] * f3 + PADE.c[8] * f4;
    U[o + n] = PADE.s[5] * f1 + PADE.s[6] * f2 + PADE.s[7] * f3 + PADE.s[8] * f4;
    CS[o] = PADE.c[0] * d + PADE.c[1] * f1 + PADE.c[2] * f2 + PADE.c[3] * f3 + PADE.c[4] * f4;
    CS[o + n] = PADE.s[0] * d + PADE.s[1] * f1 + PADE.s[2] * f2 + PADE.s[3] * f3 + PADE.s[4] * f4;
  }
}

// sK = s [Kx; Ky] (n x N)
__global__ void fold_cols_kernel(const cd* __restrict__ CS, const cd* __restrict__ kx, const cd* __restrict__ ky,
                                 int N, int batch, cd* __restrict__ sK) {
  const int n = 2 * N;
  const long long per = (long long)n * N, total = per * batch;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const long long b = e / per;
    const int rc = (int)(e % per), r = rc / N, c = rc % N;
    const cd* s = CS + b * 2ll * n * n + (long long)r * 2 * n + n;
    sK[e] = s[c] * kx[b * N + c] + s[N + c] * ky[b * N + c];
  }
}

// ------------------------------------------------------------ slice reflections
// With X = Vr^-1 tau Q s and Y = tau s P Vr:
//   even: 1 + Ge = 2 c (c + X)^-1, solved as (c + X)^T [.] = c^T
//   odd:  1 - Go = 2 (c + Y)^-1 c
// Items 0..batch of A and B get the even systems, batch..2 batch the odd ones.
// 16 x 16 tiles; the even pair is transposed through LDS.
__global__ __launch_bounds__(256) void slice_systems_kernel(const cd* __restrict__ CS, const cd* __restrict__ Cs,
                                                           const cd* __restrict__ Z, const cd* __restrict__ kx,
                                                           const cd* __restrict__ ky,
                                                           const double* __restrict__ k0d, double scale, int N,
                                                           int batch, int tiles, cd* __restrict__ A,
                                                           cd* __restrict__ B) {
  __shared__ cd ta[16][17], tb[16][17];
  const int n = 2 * N;
  const long long nn = (long long)n * n;
  const long long b = blockIdx.x / (tiles * tiles);
  const int t = blockIdx.x % (tiles * tiles);
  const int r0 = (t / tiles) * 16, c0 = (t % tiles) * 16;
  const int tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
  const int r = r0 + tr, c = c0 + tc;
  if (r < n && c < n) {
    const cd mit = mkc(0.0, -0.5 * k0d[b] * scale);  // -i tau
    const cd* cs = CS + b * 2 * nn;
    const cd cv = cs[(long long)r * 2 * n + c], sv = cs[(long long)r * 2 * n + n + c];
    const int h = r < N ? r : r - N, g = c < N ? c : c - N;
    const cd x = kx[b * N + h], y = ky[b * N + h];
    const cd so = cs[(long long)(r < N ? r + N : h) * 2 * n + n + c];
    const cd q = Cs[b * nn + (long long)r * n + c];
    const cd X = r < N ? mit * (y * y * sv - x * y * so - q) : mit * (x * x * sv - x * y * so - q);
    ta[tr][tc] = cv + X;
    tb[tr][tc] = cv;
    const cd kc = c < N ? kx[b * N + g] : ky[b * N + g];
    const cd Y = mit * (Z[b * (nn / 2) + (long long)r * N + g] * kc - sv);
    const long long o = (batch + b) * nn + (long long)r * n + c;
    A[o] = cv + Y;
    B[o] = cv;
  }
  __syncthreads();
  const int ro = c0 + tr, co = r0 + tc;
  if (ro < n && co < n) {
    const long long o = b * nn + (long long)ro * n + co;
    A[o] = ta[tc][tr];
    B[o] = tb[tc][tr];
  }
}

// S11, S12 of the slice from the solutions (even one transposed), and the
// systems of the first doubling: A = 1 -/+ S11, B = S12 for both signs.
// S holds S11, S12 in its first two blocks until the end.
__global__ __launch_bounds__(256) void slice_s_kernel(const cd* __restrict__ X, int n, int batch, int tiles,
                                                     cd* __restrict__ S, cd* __restrict__ A, cd* __restrict__ B,
                                                     int doubling) {
  __shared__ cd tx[16][17];
  const long long nn = (long long)n * n;
  const long long b = blockIdx.x / (tiles * tiles);
  const int t = blockIdx.x % (tiles * tiles);
  const int r0 = (t / tiles) * 16, c0 = (t % tiles) * 16;
  const int tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
  if (c0 + tr < n && r0 + tc < n) tx[tr][tc] = X[b * nn + (long long)(c0 + tr) * n + r0 + tc];
  __syncthreads();
  const int r = r0 + tr, c = c0 + tc;
  if (r >= n || c >= n) return;
  const long long o = (long long)r * n + c;
  const cd xe = tx[tc][tr], xo = X[(batch + b) * nn + o];
  const cd d = mkc(r == c ? 1.0 : 0.0, 0.0);
  const cd s11 = xe - xo, s12 = xe + xo - d;
  S[b * 4 * nn + o] = s11;
  S[b * 4 * nn + nn + o] = s12;
  if (doubling) {
    A[b * nn + o] = d - s11;
    A[(batch + b) * nn + o] = d + s11;
    B[b * nn + o] = s12;
    B[(batch + b) * nn + o] = s12;
  }
}

// ------------------------------------------------------------ doubling
// S11 += (E - O) / 2, S12 = (E + O) / 2 (E, O in blocks 2, 3 of S) and the next
// doubling's systems.
__global__ void doubling_kernel(cd* __restrict__ S, int n, int batch, cd* __restrict__ A, cd* __restrict__ B) {
  const long long nn = (long long)n * n, total = nn * batch;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const long long b = e / nn, o = e % nn;
    cd* sb = S + b * 4 * nn;
    const cd E = sb[2 * nn + o], O = sb[3 * nn + o];
    const cd s11 = sb[o] + 0.5 * (E - O), s12 = 0.5 * (E + O);
    const cd d = mkc((int)(o / n) == (int)(o % n) ? 1.0 : 0.0, 0.0);
    sb[o] = s11;
    sb[nn + o] = s12;
    A[b * nn + o] = d - s11;
    A[(batch + b) * nn + o] = d + s11;
    B[b * nn + o] = s12;
    B[(batch + b) * nn + o] = s12;
  }
}

// ------------------------------------------------------------ gap medium
// R1 per harmonic (a, b, c, d row-major).  kz = 0: the gap's V0 holds 1/kz and
// the reference's S-matrix is NaN there; so is this one.
__global__ void gap_reflection_kernel(const cd* __restrict__ kx, const cd* __restrict__ ky, long long total,
                                      cd* __restrict__ r1) {
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const cd x = kx[e], y = ky[e], kz = kz_gap(x, y);
    const cd k1 = mkc(1.0 + kz.x, kz.y);
    cd q = recipc(k1 * k1);
    if (kz.x == 0.0 && kz.y == 0.0) q = mkc(NAN, NAN);
    const cd a = q * (x * x - y * y), m = q * (2.0 * (x * y));
    r1[4 * e] = a;
    r1[4 * e + 1] = m;
    r1[4 * e + 2] = m;
    r1[4 * e + 3] = -a;
  }
}

// Systems (1 + G R1) Z = G for both parities; G = S11 + E | S11 - O after a
// doubling, S11 +/- S12 without one.
__global__ void gap_systems_kernel(const cd* __restrict__ S, const cd* __restrict__ r1, int N, int batch,
                                   int doubled, cd* __restrict__ A, cd* __restrict__ B) {
  const int n = 2 * N;
  const long long nn = (long long)n * n, per = (long long)n * N, total = per * batch;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const long long b = e / per;
    const int rc = (int)(e % per), r = rc / N, h = rc % N;
    const cd* q = r1 + 4 * (b * N + h);
    const cd qa = q[0], qb = q[1], qc = q[2], qd = q[3];
    const cd* sb = S + b * 4 * nn;
    const long long o1 = (long long)r * n + h, o2 = o1 + N;
    const cd s1 = sb[o1], s2 = sb[o2];
    const cd* pe = sb + (doubled ? 2 * nn : nn);
    const cd* po = sb + (doubled ? 3 * nn : nn);
    const cd d1 = mkc(r == h ? 1.0 : 0.0, 0.0), d2 = mkc(r == N + h ? 1.0 : 0.0, 0.0);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const cd g1 = p ? s1 - po[o1] : s1 + pe[o1], g2 = p ? s2 - po[o2] : s2 + pe[o2];
      const long long base = (p * (long long)batch + b) * nn;
      B[base + o1] = g1;
      B[base + o2] = g2;
      A[base + o1] = d1 + g1 * qa + g2 * qc;
      A[base + o2] = d2 + g1 * qb + g2 * qd;
    }
  }
}

struct M2 {
  cd a, b, c, d;
};
__device__ __forceinline__ M2 mul2(M2 x, M2 y) {
  return M2{x.a * y.a + x.b * y.c, x.a * y.b + x.b * y.d, x.c * y.a + x.d * y.c, x.c * y.b + x.d * y.d};
}

// G' = R1 + (1 - R1) Z (1 + R1), S11 = (Ge' + Go') / 2, S12 = (Ge' - Go') / 2
__global__ void gap_s_kernel(const cd* __restrict__ Z, const cd* __restrict__ r1, int N, int batch,
                             cd* __restrict__ S) {
  const int n = 2 * N;
  const long long nn = (long long)n * n, per = (long long)N * N, total = per * batch;
  const cd one = mkc(1.0, 0.0);
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const long long b = e / per;
    const int rc = (int)(e % per), r = rc / N, c = rc % N;
    const cd* ql = r1 + 4 * (b * N + r);
    const cd* qr = r1 + 4 * (b * N + c);
    const M2 L{one - ql[0], -ql[1], -ql[2], one - ql[3]}, R{one + qr[0], qr[1], qr[2], one + qr[3]};
    const long long o[4] = {(long long)r * n + c, (long long)r * n + N + c, (long long)(N + r) * n + c,
                            (long long)(N + r) * n + N + c};
    M2 g[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const cd* z = Z + (p * (long long)batch + b) * nn;
      g[p] = mul2(mul2(L, M2{z[o[0]], z[o[1]], z[o[2]], z[o[3]]}), R);
    }
    if (r == c) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        g[p].a = g[p].a + ql[0];
        g[p].b = g[p].b + ql[1];
        g[p].c = g[p].c + ql[2];
        g[p].d = g[p].d + ql[3];
      }
    }
    const cd ge[4] = {g[0].a, g[0].b, g[0].c, g[0].d}, go[4] = {g[1].a, g[1].b, g[1].c, g[1].d};
    cd* sb = S + b * 4 * nn;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const cd s11 = 0.5 * (ge[q] + go[q]), s12 = 0.5 * (ge[q] - go[q]);
      sb[o[q]] = s11;
      sb[nn + o[q]] = s12;
      sb[2 * nn + o[q]] = s12;
      sb[3 * nn + o[q]] = s11;
    }
  }
}

__global__ void zero_words_kernel(int* p, int count) {
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < count; e += gridDim.x * blockDim.x) p[e] = 0;
}

// info[b] = 1 for a non-finite F, -1 if any solve met an exact zero pivot, else 0
__global__ void status_kernel(const int* __restrict__ bad, const int* __restrict__ words, int batch, int nwords,
                              int* out) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  int v = bad[b];
  for (int w = 0; w < nwords; ++w)
    if (v == 0 && words[(long long)w * batch + b] != 0) v = -1;
  out[b] = v;
}

}  // namespace

int layer_scale(hipStream_t s, const cd* C, const cd* IC, long long cstride, const cd* kx, const cd* ky, int N,
                int batch, const double* k0d, double* est) {
  if (batch <= 0) return 0;
  const size_t lds = (size_t)7 * N * sizeof(cd);
  KHX_REQUIRE(lds <= 150 * 1024, "layer_scale: too many harmonics");
  KHX_TRY(ensure_dynamic_lds((const void*)layer_scale_kernel, lds));
  layer_scale_kernel<<<dim3(batch), SCALE_THREADS, lds, s>>>(C, IC, cstride, kx, ky, N, k0d, est);
  KHX_LAUNCH_CHECK();
  return 0;
}

// n^2 items: powers 4, U 2, CS 2, C s 1, s K and its product 1, A 2, B 2; the
// second right-hand sides and solutions go over U
constexpr int DIRECT_ITEMS = 14;

size_t layer_smatrix_ws_bytes(int n, int batch, int doublings) {
  return (size_t)DIRECT_ITEMS * n * n * sizeof(cd) * batch + (size_t)2 * n * sizeof(cd) * batch +
         (size_t)batch * sizeof(int) * (1 + 2 * (doublings + 2) + 2 * n) + 256;
}

int layer_smatrix(hipStream_t s, const cd* C, const cd* IC, long long cstride, const cd* kx, const cd* ky, int N,
                  int batch, const double* k0d, int doublings, cd* S, int* info, void* wsv) {
  if (batch <= 0) return 0;
  KHX_REQUIRE(doublings >= 0 && doublings <= 60, "layer_smatrix: doublings must be 0..60");
  const int n = 2 * N;
  const long long nn = (long long)n * n, NN = (long long)N * N;
  const int tiles = (n + 15) / 16;
  KHX_REQUIRE((long long)tiles * tiles * batch < (1ll << 31), "layer_smatrix: batch too large");
  cd* w = static_cast<cd*>(wsv);
  auto take = [&](long long items) {
    cd* p = w;
    w += items * nn * batch;
    return p;
  };
  cd* W4 = take(4);
  cd* U = take(2);
  cd* CS = take(2);
  cd* Cs = take(1);
  cd* half = take(1);
  cd* T = half;                     // N x 2N, then s K (n x N)
  cd* G = half + nn / 2 * batch;    // C^-1 T, then s K C^-1
  cd* A = take(2);
  cd* B = take(2);
  cd* r1 = w;
  w += 2ll * n * batch;
  int* bad = reinterpret_cast<int*>(w);
  int* words = bad + batch;
  const int nwords = 2 * (doublings + 2);
  int* perm = words + (long long)nwords * batch;
  const cd one = mkc(1.0, 0.0), zero = mkc(0.0, 0.0);
  const Mat mC{const_cast<cd*>(C), N, cstride}, mIC{const_cast<cd*>(IC), N, cstride};
  const double scale = ldexp(1.0, -doublings);

  zero_words_kernel<<<dim3((batch + 255) / 256), 256, 0, s>>>(bad, batch);
  KHX_LAUNCH_CHECK();
  // F and its powers (columns of an n x 4n buffer)
  scale_rows_kernel<<<grid_ew(NN * batch), 256, 0, s>>>(C, cstride, kx, ky, N, batch, T);
  KHX_LAUNCH_CHECK();
  KHX_TRY(zgemm(s, N, n, N, one, mIC, Mat{T, n, nn / 2}, zero, Mat{G, n, nn / 2}, batch));
  build_f_kernel<<<grid_ew(NN * batch), 256, 0, s>>>(G, C, cstride, kx, ky, k0d, scale, N, batch, W4, bad);
  KHX_LAUNCH_CHECK();
  auto power = [&](int k) { return Mat{W4 + (k - 1) * n, 4 * n, 4 * nn}; };
  KHX_TRY(zgemm(s, n, n, n, one, power(1), power(1), zero, power(2), batch));
  KHX_TRY(zgemm(s, n, 2 * n, n, one, power(2), power(1), zero, power(3), batch));  // [F^3 | F^4] = F^2 [F | F^2]
  pade_parts_kernel<<<grid_ew(nn * batch), 256, 0, s>>>(W4, n, batch, U, CS);
  KHX_LAUNCH_CHECK();
  KHX_TRY(zgemm(s, n, 2 * n, n, one, power(4), Mat{U, 2 * n, 2 * nn}, one, Mat{CS, 2 * n, 2 * nn}, batch));
  // C s (both row halves) and s K C^-1
  const Mat st{CS + n, 2 * n, 2 * nn}, sb{CS + n + (long long)N * 2 * n, 2 * n, 2 * nn};
  KHX_TRY(zgemm(s, N, n, N, one, mC, st, zero, Mat{Cs, n, nn}, batch));
  KHX_TRY(zgemm(s, N, n, N, one, mC, sb, zero, Mat{Cs + (long long)N * n, n, nn}, batch));
  fold_cols_kernel<<<grid_ew((long long)n * N * batch), 256, 0, s>>>(CS, kx, ky, N, batch, T);
  KHX_LAUNCH_CHECK();
  KHX_TRY(zgemm(s, n, N, N, one, Mat{T, N, nn / 2}, mIC, zero, Mat{G, N, nn / 2}, batch));
  // slice
  const dim3 tg((unsigned)((long long)tiles * tiles * batch));
  slice_systems_kernel<<<tg, 256, 0, s>>>(CS, Cs, G, kx, ky, k0d, scale, N, batch, tiles, A, B);
  KHX_LAUNCH_CHECK();
  const Mat mA{A, n, nn};
  KHX_TRY(zgesv_ws(s, n, n, mA, Mat{B, n, nn}, 2 * batch, perm, words));
  cd* B2 = U;
  slice_s_kernel<<<tg, 256, 0, s>>>(B, n, batch, tiles, S, A, B2, doublings > 0);
  KHX_LAUNCH_CHECK();
  const Mat s12{S + nn, n, 4 * nn};
  for (int k = 0; k < doublings; ++k) {
    if (k > 0) {
      doubling_kernel<<<grid_ew(nn * batch), 256, 0, s>>>(S, n, batch, A, B2);
      KHX_LAUNCH_CHECK();
    }
    KHX_TRY(zgesv_ws(s, n, n, mA, Mat{B2, n, nn}, 2 * batch, perm, words + 2ll * (k + 1) * batch));
    KHX_TRY(zgemm(s, n, n, n, one, s12, Mat{B2, n, nn}, zero, Mat{S + 2 * nn, n, 4 * nn}, batch));
    KHX_TRY(zgemm(s, n, n, n, one, s12, Mat{B2 + nn * batch, n, nn}, zero, Mat{S + 3 * nn, n, 4 * nn}, batch));
  }
  // gap medium
  gap_reflection_kernel<<<grid_ew((long long)N * batch), 256, 0, s>>>(kx, ky, (long long)N * batch, r1);
  KHX_LAUNCH_CHECK();
  gap_systems_kernel<<<grid_ew((long long)n * N * batch), 256, 0, s>>>(S, r1, N, batch, doublings > 0, A, B);
  KHX_LAUNCH_CHECK();
  KHX_TRY(zgesv_ws(s, n, n, mA, Mat{B, n, nn}, 2 * batch, perm, words + 2ll * (doublings + 1) * batch));
  gap_s_kernel<<<grid_ew(NN * batch), 256, 0, s>>>(B, r1, N, batch, S);
  KHX_LAUNCH_CHECK();
  if (info) {
    status_kernel<<<dim3((batch + 255) / 256), 256, 0, s>>>(bad, words, batch, nwords, info);
    KHX_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace khx
