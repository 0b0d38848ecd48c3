// Tall-skinny dense products of the reduction on gfx950: C = X^T Y (Gram
// matrices, reorthogonalisation and reduced matrices), Y = alpha Y + beta X S
// (block updates, Ritz vectors, recovery) and the Cholesky factor of the
// Lanczos block's Gram matrix.  X and Y are row-major with their own leading
// dimensions.  All products run on FP64 MFMA with operands straight from
// memory; every sum has a fixed order.
#include <algorithm>
#include "kern_device.hpp"

namespace fgpu {

// ---------------------------------------------------------------- X^T Y
// One workgroup: 16 XA columns of X by 16 YB columns of Y over crows rows,
// split over its WV waves in whole groups of four rows (one MFMA step).
// Lane (lr, lk) of a step takes row lk of the group and column lr of either
// operand: 128 contiguous bytes per row and 16 columns.  The waves' sums are
// added in wave order through LDS.  Output: the chunk's partial matrix
// part[chunk][a][b], or with one chunk C itself (and acc, see launch_xty).
// Rows past the range repeat the last one with a zero X operand, columns
// past it repeat the last one and are dropped.  lower: tiles wholly above the
// diagonal of C are left out (117x109 plate, 384 x 384: 557 -> 334 us; 480 with a chunk's tiles spread over the XCDs).
// Bound by HBM for tall X (one read of X and Y), by its own latency below
// some thousand rows, where one workgroup per column tile needs no second
// launch for the sum: 64 columns x 16 over 354 rows 15 -> 8 us, 16 x 16 6 us,
// the Lanczos block against up to 128 basis vectors of 45,864 rows 34 -> 26
// us on average.
template <int XA, int YB, int WV>
__global__ __launch_bounds__(64 * WV) void k_xty(int n, int crows, int na, int nb, const double* __restrict__ X,
                                                 int ldx, const double* __restrict__ Y, int ldy,
                                                 double* __restrict__ part, double* __restrict__ C,
                                                 double* __restrict__ acc_out, int acc_add, int nta, int ntile,
                                                 int lower) {
  constexpr int ST = XA * YB == 1 ? 8 : XA * YB <= 4 ? 4 : 2;  // steps in flight
  constexpr int TS = 16 * YB + 1;                               // LDS tile row
  __shared__ double red[16 * XA * TS];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  // the tiles of a chunk of rows are neighbours on one XCD and read them
  // through its L2; lower: tile q of the lower triangle in row order
  const int id = xcd_ranges(blockIdx.x, gridDim.x), chunk = id / ntile;
  int ta = id % ntile, tb = 0;
  if (lower) {
    int row = 0;
    while (ta > row) ta -= ++row;
    tb = ta;
    ta = row;
  } else {
    tb = ta / nta;
    ta %= nta;
  }
  const int a0 = 16 * XA * ta, b0 = 16 * YB * tb;
  const int c0 = chunk * crows, rows = min(crows, n - c0);
  const int per = ((rows + 4 * WV - 1) / (4 * WV)) * 4;  // rows per wave
  const int rb = min(rows, wv * per), re = min(rows, rb + per);
  const double *xp[XA], *yp[YB];
#pragma unroll
  for (int x = 0; x < XA; x++) xp[x] = X + (int64_t)c0 * ldx + min(a0 + 16 * x + lr, na - 1);
#pragma unroll
  for (int y = 0; y < YB; y++) yp[y] = Y + (int64_t)c0 * ldy + min(b0 + 16 * y + lr, nb - 1);
  f64x4 acc[XA][YB];
#pragma unroll
  for (int x = 0; x < XA; x++)
#pragma unroll
    for (int y = 0; y < YB; y++) acc[x][y] = f64x4{0.0, 0.0, 0.0, 0.0};
  struct Stage {
    double x[ST][XA], y[ST][YB];
  };
  auto load = [&](int r0, Stage& g) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const int64_t r = min(r0 + 4 * s + lk, re - 1);
#pragma unroll
      for (int x = 0; x < XA; x++) g.x[s][x] = xp[x][r * ldx];
#pragma unroll
      for (int y = 0; y < YB; y++) g.y[s][y] = yp[y][r * ldy];
    }
  };
  auto multiply = [&](int r0, const Stage& g) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const bool in = r0 + 4 * s + lk < re;
#pragma unroll
      for (int x = 0; x < XA; x++)
#pragma unroll
        for (int y = 0; y < YB; y++)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(g.y[s][y], in ? g.x[s][x] : 0.0, acc[x][y], 0, 0, 0);
    }
  };
  if (rb < re) {
    Stage g0, g1;
    load(rb, g0);
    for (int r = rb; r < re; r += 8 * ST) {
      if (r + 4 * ST < re) load(r + 4 * ST, g1);
      multiply(r, g0);
      if (r + 4 * ST >= re) break;
      if (r + 8 * ST < re) load(r + 8 * ST, g0);
      multiply(r + 4 * ST, g1);
    }
  }
  // acc[x][y][q]: column 16 x + lr of X, column 16 y + lk + 4 q of Y
  for (int w = 0; w < WV; w++) {
    if (wv == w) {
#pragma unroll
      for (int x = 0; x < XA; x++)
#pragma unroll
        for (int y = 0; y < YB; y++)
#pragma unroll
          for (int q = 0; q < 4; q++) {
            double& t = red[(16 * x + lr) * TS + 16 * y + lk + 4 * q];
            t = w == 0 ? acc[x][y][q] : t + acc[x][y][q];
          }
    }
    __syncthreads();
  }
  const bool whole = (int)gridDim.x == ntile;
  double* P = whole ? C : part + (int64_t)chunk * na * nb;
  for (int e = threadIdx.x; e < 256 * XA * YB; e += 64 * WV) {
    const int a = e / (16 * YB), b = e % (16 * YB);
    if (a0 + a >= na || b0 + b >= nb) continue;
    const int64_t o = (int64_t)(a0 + a) * nb + b0 + b;
    const double v = red[a * TS + b];
    P[o] = v;
    if (whole && acc_out) acc_out[o] = acc_add ? acc_out[o] + v : v;
  }
}

// C = the sum of the chunk partials; acc (optional) = C, or acc + C with
// acc_add.  64 entries per workgroup; wave w adds chunks w, w + 4, ... in
// order, then the four waves' sums are added in wave order.
__global__ __launch_bounds__(256) void k_xty_sum(int nchunk, int nab, const double* __restrict__ part,
                                                 double* __restrict__ C, double* __restrict__ acc, int acc_add) {
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, e = blockIdx.x * 64 + lane;
  const double* p = part + min(e, nab - 1);
  double s = 0.0;
  int c = wv;
  for (; c + 28 < nchunk; c += 32) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = p[(int64_t)(c + 4 * u) * nab];
#pragma unroll
    for (int u = 0; u < 8; u++) s += v[u];
  }
  for (; c < nchunk; c += 4) s += p[(int64_t)c * nab];
  red[wv][lane] = s;
  __syncthreads();
  if (wv == 0 && e < nab) {
    const double v = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
    C[e] = v;
    if (acc) acc[e] = acc_add ? acc[e] + v : v;
  }
}

// Row chunks of X^T Y: the callers' bound on the partial matrices.
int xty_chunks(int n) { return (n + 127) / 128; }

template <int XA, int YB, int WV>
static int xty_go(hipStream_t st, int n, int na, int nb, const double* X, int ldx, const double* Y, int ldy,
                  double* part, double* C, double* acc, int acc_add, int lower) {
  // chunks of about 32 rows a wave at most, more where that would make more
  // workgroups than fill the 256 CUs a few times over (each chunk costs a
  // partial matrix)
  const int ta = (int)nblk(na, 16 * XA), tb = (int)nblk(nb, 16 * YB);
  if (XA != YB || na != nb) lower = 0;
  const int tiles = lower ? ta * (ta + 1) / 2 : ta * tb;
  const int most = std::max(1, 2048 / WV / tiles), crows0 = 32 * WV;
  int nch = std::min(most, std::max(1, (n + crows0 - 1) / crows0));
  const int crows = (n + nch - 1) / nch;
  nch = (n + crows - 1) / crows;
  k_xty<XA, YB, WV><<<nch * tiles, 64 * WV, 0, st>>>(n, crows, na, nb, X, ldx, Y, ldy, part, C, acc, acc_add, ta, tiles,
                                                     lower);
  return nch;
}

void launch_xty(hipStream_t st, int n, int na, int nb, const double* X, int ldx, const double* Y, int ldy,
                double* part, double* C, double* acc, bool acc_add, bool sym) {
  if (na <= 0 || nb <= 0) return;
  if (n <= 0) {
    launch_fill(st, C, (int64_t)na * nb, 0.0);
    if (acc && !acc_add) launch_fill(st, acc, (int64_t)na * nb, 0.0);
    return;
  }
  const int add = acc_add ? 1 : 0, lower = sym ? 1 : 0;
  int nch = 0;
  // tiles: as wide as the operands, 64 x 64 at most; the waves of a narrow
  // one split the rows 16 ways
  if (nb <= 16) {
    if (na <= 16) nch = xty_go<1, 1, 16>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
    else if (na <= 32) nch = xty_go<2, 1, 16>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
    else nch = xty_go<4, 1, 8>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
  } else if (nb <= 32) {
    if (na <= 32) nch = xty_go<2, 2, 8>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
    else nch = xty_go<4, 2, 4>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
  } else {
    if (na <= 16) nch = xty_go<1, 4, 8>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
    else if (na <= 32) nch = xty_go<2, 4, 4>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
    else nch = xty_go<4, 4, 4>(st, n, na, nb, X, ldx, Y, ldy, part, C, acc, add, lower);
  }
  if (nch > 1) k_xty_sum<<<nblk((int64_t)na * nb, 64), 256, 0, st>>>(nch, na * nb, part, C, acc, add);
}

// ---------------------------------------------------------------- X S
// Y = alpha Y + beta X S for S with at most 16 NB columns, one wave per 16 RT
// rows.  A load takes 32 neighbouring columns of two rows; the wave turns its
// 16 x 32 chunks through its own LDS tiles into the MFMA operand, one chunk
// ahead of the products (step s multiplies k = 8 (lane / 16) + s).  RT = 2
// where there are rows for it: the S operand, as many bytes as X per 16 rows,
// is then read once for 32.  blockIdx.y = 1 takes the second pair (X2, Y2)
// with the same S; dup (optional) gets a copy of the second pair's result.  Y
// may be X (a wave has read its rows before it writes them).  Bound by HBM.
template <int NB, int RT>
__global__ __launch_bounds__(256) void k_xs(int n, int na, int nb, const double* X1, int ldx1,
                                            const double* __restrict__ Sm, double* Y1, int ldy1, double alpha,
                                            double beta, const double* X2, int ldx2, double* Y2, int ldy2,
                                            double* __restrict__ dup, int ldd) {
  constexpr int LT = 34;  // tile element (row, k) at row LT + 4 (k mod 8) + k / 8: conflict-free reads
  __shared__ double tiles[4][RT][16 * LT];
  const double* X = blockIdx.y ? X2 : X1;
  double* Y = blockIdx.y ? Y2 : Y1;
  const int ldx = blockIdx.y ? ldx2 : ldx1, ldy = blockIdx.y ? ldy2 : ldy1;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int r0 = 16 * RT * (4 * blockIdx.x + wv);
  if (r0 >= n) return;
  const int ka = lane & 31, ia = lane >> 5;
  // row r0 + 2 q + ia of X, q < 8 RT (rows past the end repeat the last one)
  const double* xb = X + (int64_t)r0 * ldx;
  int64_t xo[8 * RT];
#pragma unroll
  for (int q = 0; q < 8 * RT; q++) xo[q] = (int64_t)min(2 * q + ia, n - 1 - r0) * ldx;
  int col[NB];
#pragma unroll
  for (int y = 0; y < NB; y++) col[y] = min(16 * y + lr, nb - 1);
  f64x4 acc[RT][NB];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int y = 0; y < NB; y++) acc[t][y] = f64x4{0.0, 0.0, 0.0, 0.0};
  double x[8 * RT], s[2][8][NB];
  auto load_x = [&](int k0) {
    const double* p = xb + min(k0 + ka, na - 1);
#pragma unroll
    for (int q = 0; q < 8 * RT; q++) x[q] = p[xo[q]];
  };
  auto load_s = [&](int k0, double (&g)[8][NB]) {
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const double* p = Sm + (int64_t)min(k0 + 8 * lk + m, na - 1) * nb;
#pragma unroll
      for (int y = 0; y < NB; y++) g[m][y] = p[col[y]];
    }
  };
  auto chunk = [&](int k0, double (&cur)[8][NB], double (&nxt)[8][NB]) {
    const bool in = k0 + ka < na;
#pragma unroll
    for (int q = 0; q < 8 * RT; q++)
      tiles[wv][q / 8][(2 * (q % 8) + ia) * LT + 4 * (ka & 7) + (ka >> 3)] = in ? x[q] : 0.0;
    if (k0 + 32 < na) {
      load_x(k0 + 32);
      load_s(k0 + 32, nxt);
    }
    __builtin_amdgcn_wave_barrier();  // the tiles are this wave's own: LDS keeps its order
#pragma unroll
    for (int m = 0; m < 8; m++)
#pragma unroll
      for (int t = 0; t < RT; t++) {
        const double xv = tiles[wv][t][lr * LT + 4 * m + lk];
#pragma unroll
        for (int y = 0; y < NB; y++)
          acc[t][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur[m][y], xv, acc[t][y], 0, 0, 0);
      }
    __builtin_amdgcn_wave_barrier();
  };
  if (na > 0) {
    load_x(0);
    load_s(0, s[0]);
    for (int k0 = 0; k0 < na; k0 += 64) {
      chunk(k0, s[0], s[1]);
      if (k0 + 32 < na) chunk(k0 + 32, s[1], s[0]);
    }
  }
  // acc[t][y][q]: row r0 + 16 t + lr, column 16 y + lk + 4 q
#pragma unroll
  for (int t = 0; t < RT; t++) {
    const int r = r0 + 16 * t + lr;
    if (r >= n) continue;
    double* out = Y + (int64_t)r * ldy;
#pragma unroll
    for (int y = 0; y < NB; y++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int j = 16 * y + lk + 4 * q;
        if (j >= nb) continue;
        const double v = ((alpha == 0.0) ? 0.0 : alpha * out[j]) + beta * acc[t][y][q];
        out[j] = v;
        if (dup && blockIdx.y) dup[(int64_t)r * ldd + j] = v;
      }
  }
}

// Y[r][j] = alpha*Y[r][j] + beta * sum_a X[r][a] S[a][j]; S is (na x nb) row-major.
__global__ __launch_bounds__(256) void k_gemm_small(int n, int na, int nb, const double* __restrict__ X,
                                                    int ldx, const double* __restrict__ Sm,
                                                    double* __restrict__ Y, int ldy, double alpha,
                                                    double beta) {
  extern __shared__ double sS[];
  for (int i = threadIdx.x; i < na * nb; i += blockDim.x) sS[i] = Sm[i];
  __syncthreads();
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int r = (int)(g / nb), j = (int)(g % nb);
  if (r >= n) return;
  double s = 0.0;
  for (int a = 0; a < na; a++) s += X[(int64_t)r * ldx + a] * sS[a * nb + j];
  double y = (alpha == 0.0) ? 0.0 : alpha * Y[(int64_t)r * ldy + j];
  Y[(int64_t)r * ldy + j] = y + beta * s;
}

static void xs_go(hipStream_t st, int n, int na, int nb, const double* X1, int ldx1, const double* Sm, double* Y1,
                  int ldy1, double alpha, double beta, const double* X2, int ldx2, double* Y2, int ldy2, double* dup,
                  int ldd) {
  // 32 rows a wave once that still gives every SIMD a wave (1024 waves)
  const bool tall = n >= 32768 && nb <= 32;
  const dim3 g(nblk(n, tall ? 128 : 64), X2 ? 2 : 1);
  auto go = [&](auto nbt, auto rt) {
    k_xs<decltype(nbt)::value, decltype(rt)::value><<<g, 256, 0, st>>>(n, na, nb, X1, ldx1, Sm, Y1, ldy1, alpha, beta, X2,
                                                                       ldx2, Y2, ldy2, dup, ldd);
  };
  using std::integral_constant;
  if (nb <= 16) tall ? go(integral_constant<int, 1>{}, integral_constant<int, 2>{}) : go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
  else if (nb <= 32) tall ? go(integral_constant<int, 2>{}, integral_constant<int, 2>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  else if (nb <= 48) go(integral_constant<int, 3>{}, integral_constant<int, 1>{});
  else go(integral_constant<int, 4>{}, integral_constant<int, 1>{});
}

void launch_gemm_small2(hipStream_t st, int n, int na, int nb, const double* X1, int ldx1, double* Y1, int ldy1,
                        const double* X2, int ldx2, double* Y2, int ldy2, const double* Sm, double* dup, int ldd) {
  if (n > 0 && nb > 0) xs_go(st, n, na, nb, X1, ldx1, Sm, Y1, ldy1, 0.0, 1.0, X2, ldx2, Y2, ldy2, dup, ldd);
}

void launch_gemm_small(hipStream_t st, int n, int na, int nb, const double* X, int ldx, const double* Sm,
                       double* Y, int ldy, double alpha, double beta) {
  if (n <= 0 || nb <= 0) return;
  if (nb <= 64) {
    xs_go(st, n, na, nb, X, ldx, Sm, Y, ldy, alpha, beta, nullptr, 0, nullptr, 0, nullptr, 0);
    return;
  }
  // S is staged in LDS in row chunks of at most 64 KiB; chunk k adds
  // beta X_k S_k to the result of the chunks before it (fixed order)
  const int rows = std::max(1, (int)(65536 / (sizeof(double) * nb)));
  for (int a0 = 0; a0 < na || a0 == 0; a0 += rows) {
    const int ka = std::min(rows, na - a0);
    k_gemm_small<<<nblk((int64_t)n * nb, 256), 256, sizeof(double) * std::max(ka, 1) * nb, st>>>(
        n, ka, nb, X + a0, ldx, Sm + (size_t)a0 * nb, Y, ldy, a0 == 0 ? alpha : 1.0, beta);
    if (na <= 0) break;
  }
}

// ---------------------------------------------------------------- Gram matrix factor
// Cholesky factor of the symmetrised n x n Gram matrix G = R^T R (R upper,
// row-major) and R^{-1}, by one workgroup (n <= 64): at step j every thread
// forms the pivot (same value in each), thread i > j the entry R[j][i]; the
// inverse is solved column by column, thread t owning column t.  *bad = 1
// for a non-positive pivot (the block has broken down), else 0 if first.
__global__ __launch_bounds__(64) void k_chol_inv(int n, const double* __restrict__ G, double* __restrict__ R,
                                                 double* __restrict__ Ri, int first, int* __restrict__ bad) {
  __shared__ double A[64][65], U[64][65], V[64][65];
  const int t = threadIdx.x;
  if (t < n)
    for (int i = 0; i < n; i++) {
      A[i][t] = i == t ? G[i * n + t] : 0.5 * (G[i * n + t] + G[t * n + i]);
      U[i][t] = 0.0;
      V[i][t] = 0.0;
    }
  bool nonpos = false;
  __syncthreads();
  for (int j = 0; j < n; j++) {
    double s = A[j][j];
    for (int k = 0; k < j; k++) s -= U[k][j] * U[k][j];
    if (!(s > 0.0)) {
      nonpos = true;
      s = 1.0;
    }
    const double d = sqrt(s);
    if (t == j) U[j][j] = d;
    if (t > j && t < n) {
      double v = A[j][t];
      for (int k = 0; k < j; k++) v -= U[k][j] * U[k][t];
      U[j][t] = v / d;
    }
    __syncthreads();
  }
  if (t == 0 && (first || nonpos)) *bad = nonpos ? 1 : 0;
  if (t < n) {
    V[t][t] = 1.0 / U[t][t];
    for (int i = t - 1; i >= 0; i--) {
      double v = 0.0;
      for (int k = i + 1; k <= t; k++) v += U[i][k] * V[k][t];
      V[i][t] = -v / U[i][i];
    }
    for (int i = 0; i < n; i++) {
      R[i * n + t] = U[i][t];
      Ri[i * n + t] = V[i][t];
    }
  }
}

// k_chol_inv for n <= 16, adding up the nch chunk partials of G first (1024
// threads: four groups of chunks per entry).  One wave then has the rows in
// registers: lane i < 16 holds row i and lane 16 + i row i of the identity,
// so the LDL^T sweep (readlane broadcasts, one reciprocal per pivot, as in
// the fronts' diagonal blocks) gives the unit lower L1, D and X1 = L1^-1;
// G = R^T R with R = D^1/2 L1^T and R^-1 = X1^T D^-1/2.  Rows and columns
// beyond n are identity.  A chain of 16 pivots: 9.5 + 4 us for the sum of the
// partials -> 5.6 us with one chunk, 9.5 with 128.
__global__ __launch_bounds__(1024) void k_chol16(int n, int nch, const double* __restrict__ part,
                                                 double* __restrict__ R, double* __restrict__ Ri, int first,
                                                 int* __restrict__ bad) {
  __shared__ double sG[4][16][17], sS[16][17];
  {
    const int e = threadIdx.x & 255, g = threadIdx.x >> 8, i = e >> 4, m = e & 15;
    double s = 0.0;
    if (i < n && m < n) {
      const double* q = part + i * n + m;
      const int64_t step = (int64_t)n * n;
      int c = g;
      for (; c + 28 < nch; c += 32) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = q[(c + 4 * u) * step];
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
      }
      for (; c < nch; c += 4) s += q[c * step];
    } else if (g == 0) {
      s = i == m ? 1.0 : 0.0;
    }
    sG[g][i][m] = s;
  }
  __syncthreads();
  if (threadIdx.x < 256) {
    const int i = threadIdx.x >> 4, m = threadIdx.x & 15;
    auto gram = [&](int r, int c) { return ((sG[0][r][c] + sG[1][r][c]) + sG[2][r][c]) + sG[3][r][c]; };
    sS[i][m] = 0.5 * (gram(i, m) + gram(m, i));
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x, row = lane & 15, unit = lane - 16;
  double a[16], u[16];
#pragma unroll
  for (int m = 0; m < 16; m++) a[m] = unit < 0 ? sS[row][m] : (unit == m ? 1.0 : 0.0);
  // a non-positive pivot goes on as 1 (a select per pivot on its own lane)
  bool nonpos = lane == 0 && !(a[0] > 0.0);
  auto pivot = [&](double v, int j) { return lane_bcast(v > 0.0 ? v : 1.0, j); };
  double dj = pivot(a[0], 0), rj = recip64(dj);
#pragma unroll
  for (int j = 0; j < 16; j++) {
    u[j] = a[j];
    double ub[16];
#pragma unroll
    for (int m = j + 1; m < 16; m++) ub[m] = lane_bcast(u[j], m);
    const double q = u[j] * rj, l = __builtin_fma(__builtin_fma(-dj, q, u[j]), rj, q);
    a[j] = lane > j ? l : (lane == j ? dj : a[j]);
    if (j == 15) break;
    __builtin_amdgcn_sched_barrier(0);
    a[j + 1] = __builtin_fma(-l, ub[j + 1], a[j + 1]);
    nonpos = nonpos || (lane == j + 1 && !(a[j + 1] > 0.0));
    dj = pivot(a[j + 1], j + 1);
    rj = recip64(dj);
#pragma unroll
    for (int m = j + 2; m < 16; m++) a[m] = __builtin_fma(-l, ub[m], a[m]);
    __builtin_amdgcn_sched_barrier(0);
  }
  nonpos = __any(nonpos);
  if (lane == 0 && (first || nonpos)) *bad = nonpos ? 1 : 0;
  // lane i < 16: D_i = a[i], L1[i][m] = a[m] (m < i); lane 16 + i: X1[m][i] = u[m]
  double di = a[0];
#pragma unroll
  for (int m = 1; m < 16; m++) di = m == lane ? a[m] : di;
  const double sd = sqrt(lane < 16 ? di : 1.0), rs = 1.0 / sd;
  // R[m][i] = sqrt(D_m) L1[i][m] (m < i), sqrt(D_i) on the diagonal, 0 above;
  // R^-1[i][m] = X1[m][i] / sqrt(D_m) (m >= i), 0 below: through LDS, then
  // one store per entry
#pragma unroll
  for (int m = 0; m < 16; m++) {
    const double sm = lane_bcast(sd, m), rm = lane_bcast(rs, m);
    if (lane < 16) sG[0][m][lane] = m < lane ? sm * a[m] : (m == lane ? sd : 0.0);
    else if (unit < 16) sG[1][unit][m] = m >= unit ? u[m] * rm : 0.0;
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int e = lane; e < 256; e += 64) {
    const int i = e >> 4, m = e & 15;
    if (i < n && m < n) {
      R[i * n + m] = sG[0][i][m];
      Ri[i * n + m] = sG[1][i][m];
    }
  }
}

void launch_gram_inv(hipStream_t st, int n, int bs, const double* X, const double* Y, double* part, double* G,
                     double* R, double* Ri, bool first, int* bad) {
  const int f = first ? 1 : 0;
  if (bs <= 16) {
    const int nch = xty_go<1, 1, 16>(st, n, bs, bs, X, bs, Y, bs, part, G, nullptr, 0, 0);
    k_chol16<<<1, 1024, 0, st>>>(bs, nch, nch > 1 ? part : G, R, Ri, f, bad);
  } else {
    launch_xty(st, n, bs, bs, X, bs, Y, bs, part, G);
    k_chol_inv<<<1, 64, 0, st>>>(bs, G, R, Ri, f, bad);
  }
}

}  // namespace fgpu
