// gfx950 kernels of the part reducer: element matrices, pull assembly,
// multifrontal LDL^T (pivot sweeps in registers, everything else of a diagonal
// block, the panels and the trailing updates on MFMA) and sparse products; the
// triangular solves are in solve.hip, the tall-skinny products in dense.hip.
//
// Front storage: the front of supernode s is an nrow x nrow column-major
// FP64 block at pool + foff[s]; only its lower triangle is meaningful.  After
// factorisation its first ncol columns hold L (unit diagonal implied) with D
// on the diagonal, and the trailing (nrow-ncol)^2 block holds the update
// (contribution) matrix the parent adds in.
#include <algorithm>
#include <climits>
#include <type_traits>
#include "kern_device.hpp"

namespace fgpu {

// ---------------------------------------------------------------- HEX8
// One 64-lane workgroup per element.  Lanes 0..26 evaluate the 27 Gauss
// points (Femlib/hexa.f HEXA31 with NIP=3 and HEXA35/PRIMAS share the same
// 3x3x3 rule, whose abscissa and weights are single-precision literals in
// the Fortran source), lanes 0..35 then accumulate one 3x3 node-pair block
// of K and of the consistent M each.
__global__ __launch_bounds__(64) void k_hex8(int nhex, const int* __restrict__ elist,
                                             const int* __restrict__ eptr,
                                             const int* __restrict__ enodes,
                                             const double* __restrict__ xyz,
                                             const double* __restrict__ eprop,
                                             const int64_t* __restrict__ eoff,
                                             double* __restrict__ Kp, double* __restrict__ Mp,
                                             int* __restrict__ ebad) {
  __shared__ double sX[3][8];
  __shared__ double sD[27][24];  // dN/dx: [n*8 + node]
  __shared__ double sN[27][8];
  __shared__ double sW[27];
  __shared__ int sBad;
  const int lane = threadIdx.x;
  const int e = elist[blockIdx.x];
  if (lane == 0) sBad = 0;
  if (lane < 24) {
    int node = enodes[eptr[e] + (lane & 7)];
    sX[lane >> 3][lane & 7] = xyz[3 * node + (lane >> 3)];
  }
  __syncthreads();
  const double a3 = (double)0.77459666924148f;
  const double wt1 = (double)0.55555555555556f, wt2 = (double)0.88888888888889f;
  const double* X = sX[0];
  const double* Y = sX[1];
  const double* Z = sX[2];
  auto jac = [&](double xi, double eta, double zeta, double* BJ, bool inv) -> double {
    double A1 = 1. + xi, A2 = 1. - xi, B1 = 1. + eta, B2 = 1. - eta, C1 = 1. + zeta, C2 = 1. - zeta;
    double J[3][3];
    const double* V[3] = {X, Y, Z};
    for (int c = 0; c < 3; c++) {
      const double* v = V[c];
      J[0][c] = 0.125 * (B1 * C1 * (v[6] - v[7]) - B2 * C1 * (v[4] - v[5]) + B1 * C2 * (v[2] - v[3]) - B2 * C2 * (v[0] - v[1]));
      J[1][c] = 0.125 * (A1 * C1 * (v[6] - v[5]) + A2 * C1 * (v[7] - v[4]) + A1 * C2 * (v[2] - v[1]) + A2 * C2 * (v[3] - v[0]));
      J[2][c] = 0.125 * (A1 * B1 * (v[6] - v[2]) + A2 * B1 * (v[7] - v[3]) + A2 * B2 * (v[4] - v[0]) + A1 * B2 * (v[5] - v[1]));
    }
    double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) - J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                 J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    if (inv)
      for (int q = 0; q < 9; q++) BJ[q] = 0.0;  // hexa.f:814-816 zeroes BJ first
    if (inv && det > 0.0) {
      double r = 1. / det;
      BJ[0] = r * (J[1][1] * J[2][2] - J[2][1] * J[1][2]);
      BJ[1] = -r * (J[0][1] * J[2][2] - J[0][2] * J[2][1]);
      BJ[2] = r * (J[0][1] * J[1][2] - J[0][2] * J[1][1]);
      BJ[3] = -r * (J[1][0] * J[2][2] - J[1][2] * J[2][0]);
      BJ[4] = r * (J[0][0] * J[2][2] - J[0][2] * J[2][0]);
      BJ[5] = -r * (J[0][0] * J[1][2] - J[0][2] * J[1][0]);
      BJ[6] = r * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
      BJ[7] = -r * (J[0][0] * J[2][1] - J[0][1] * J[2][0]);
      BJ[8] = r * (J[0][0] * J[1][1] - J[0][1] * J[1][0]);
    }
    return det;
  };
  if (lane < 27) {
    int ix = lane % 3, iy = (lane / 3) % 3, iz = lane / 9;
    double gp[3] = {-a3, 0.0, a3}, gw[3] = {wt1, wt2, wt1};
    double xi = gp[ix], eta = gp[iy], zeta = gp[iz];
    double BJ[9];
    double det = jac(xi, eta, zeta, BJ, true);
    sW[lane] = gw[ix] * gw[iy] * gw[iz] * det;
    double xip = 1. + xi, xim = 1. - xi, etap = 1. + eta, etam = 1. - eta, zetp = 1. + zeta, zetm = 1. - zeta;
    for (int n = 0; n < 3; n++) {
      // BJ row n = (BJ(n,1), BJ(n,2), BJ(n,3)) of the Fortran inverse Jacobian
      double b1 = BJ[3 * n + 0], b2 = BJ[3 * n + 1], b3 = BJ[3 * n + 2];
      double* D = &sD[lane][n * 8];
      D[0] = .125 * (-b1 * etam * zetm - b2 * xim * zetm - b3 * xim * etam);
      D[1] = .125 * (b1 * etam * zetm - b2 * xip * zetm - b3 * xip * etam);
      D[2] = .125 * (b1 * etap * zetm + b2 * xip * zetm - b3 * xip * etap);
      D[3] = .125 * (-b1 * etap * zetm + b2 * xim * zetm - b3 * xim * etap);
      D[4] = .125 * (-b1 * etam * zetp - b2 * xim * zetp + b3 * xim * etam);
      D[5] = .125 * (b1 * etam * zetp - b2 * xip * zetp + b3 * xip * etam);
      D[6] = .125 * (b1 * etap * zetp + b2 * xip * zetp + b3 * xip * etap);
      D[7] = .125 * (-b1 * etap * zetp + b2 * xim * zetp + b3 * xim * etap);
    }
    sN[lane][0] = .125 * xim * etam * zetm;
    sN[lane][1] = .125 * xip * etam * zetm;
    sN[lane][2] = .125 * xip * etap * zetm;
    sN[lane][3] = .125 * xim * etap * zetm;
    sN[lane][4] = .125 * xim * etam * zetp;
    sN[lane][5] = .125 * xip * etam * zetp;
    sN[lane][6] = .125 * xip * etap * zetp;
    sN[lane][7] = .125 * xim * etap * zetp;
  } else if (lane < 35) {
    // Jacobian sign check at the nodes (hexa.f:75-80)
    const double cx[8] = {-1, 1, 1, -1, -1, 1, 1, -1}, cy[8] = {-1, -1, 1, 1, -1, -1, 1, 1},
                 cz[8] = {-1, -1, -1, -1, 1, 1, 1, 1};
    int i = lane - 27;
    if (jac(cx[i], cy[i], cz[i], nullptr, false) < 0.0) sBad = 1;
  }
  __syncthreads();
  if (lane == 0 && sBad) ebad[e] = -2;
  if (lane >= 36) return;
  const double E = eprop[NPROP * e + P_E], nu = eprop[NPROP * e + P_NU], rho = eprop[NPROP * e + P_RHO];
  const double fac = E / ((1.0 + nu) * (1.0 - nu - nu));
  const double C11 = (1.0 - nu) * fac, C12 = nu * fac, G = (0.5 - nu) * fac;
  int a = (int)((sqrt(8.0 * lane + 1.0) - 1.0) * 0.5);
  while ((a + 1) * (a + 2) / 2 <= lane) a++;
  while (a * (a + 1) / 2 > lane) a--;
  const int b = lane - a * (a + 1) / 2;
  double acc[9], macc = 0.0;
#pragma unroll
  for (int q = 0; q < 9; q++) acc[q] = 0.0;
  for (int g = 0; g < 27; g++) {
    double da[3] = {sD[g][a], sD[g][8 + a], sD[g][16 + a]};
    double db[3] = {sD[g][b], sD[g][8 + b], sD[g][16 + b]};
    double wd = sW[g];
    double dot = da[0] * db[0] + da[1] * db[1] + da[2] * db[2];
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        double v = (r == c) ? C11 * da[r] * db[r] + G * (dot - da[r] * db[r])
                            : C12 * da[r] * db[c] + G * da[c] * db[r];
        acc[3 * r + c] += wd * v;
      }
    macc += wd * sN[g][a] * sN[g][b];
  }
  const int64_t off = eoff[e] + 9 * lane;
#pragma unroll
  for (int q = 0; q < 9; q++) {
    Kp[off + q] = acc[q];
    Mp[off + q] = (q % 4 == 0) ? rho * macc : 0.0;
  }
}

// ---------------------------------------------------------------- assembly
// Owner-computes (pull) assembly: every CSR entry sums its element
// contributions in a fixed order, so the result is deterministic and needs no
// atomics or colouring passes.  Lower-triangle stiffness entries are also
// written straight into their front position.
template <bool COEF>
__global__ __launch_bounds__(256) void k_assemble(int64_t nnz, const int* __restrict__ cptr,
                                                  const int* __restrict__ cidx,
                                                  const double* __restrict__ ccoef,
                                                  const double* __restrict__ Kp,
                                                  const double* __restrict__ Mp,
                                                  double* __restrict__ Kv, double* __restrict__ Mv,
                                                  const int64_t* __restrict__ fmap,
                                                  double* __restrict__ pool) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  double kv = 0.0, mv = 0.0;
  for (int q = cptr[k]; q < cptr[k + 1]; q++) {
    const int c = cidx[q];
    if (COEF) {  // rigid-element constraint coefficient of this contribution
      const double w = ccoef[q];
      kv += w * Kp[c];
      mv += w * Mp[c];
    } else {
      kv += Kp[c];
      mv += Mp[c];
    }
  }
  Kv[k] = kv;
  Mv[k] = mv;
  if (pool) {  // FP64 factor: original entries straight into the fronts
    int64_t f = fmap[k];
    if (f >= 0) pool[f] = kv;
  }
}

// original diagonal a_jj of the first n permuted equations (times rs_j^2 when
// rs is given: the equilibrated matrix) and the largest |a_jj| in *amax
// (non-negative doubles order as their bit patterns; *amax starts at 0).  One
// atomic per workgroup: one per thread on the one address, and a walk along
// the row to its diagonal, took 14 us for 354 rows and 48 for 77,496 (now 4 and 6).
__global__ __launch_bounds__(256) void k_diag_extract(int n, const int* __restrict__ dpos,
                                                      const double* __restrict__ val, const double* __restrict__ rs,
                                                      double* __restrict__ adiag, unsigned long long* __restrict__ amax) {
  __shared__ double top[4];
  double big = 0.0;
  for (int r = blockIdx.x * 256 + threadIdx.x; r < n; r += gridDim.x * 256) {
    double a = val[dpos[r]];
    if (rs) a *= rs[r] * rs[r];
    adiag[r] = a;
    big = fabs(a) > big ? fabs(a) : big;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) big = fmax(big, __shfl_xor(big, off));
  if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = big;
  __syncthreads();
  if (threadIdx.x == 0)
    atomicMax(amax, (unsigned long long)__double_as_longlong(fmax(fmax(top[0], top[1]), fmax(top[2], top[3]))));
}

// Start values of a reduction, in one launch: no element and no pivot flagged,
// the pivot statistics below, *amax = 0.
__global__ __launch_bounds__(256) void k_begin(int nel, int* __restrict__ ebad, int n, int* __restrict__ sing,
                                               int* __restrict__ stats, double* __restrict__ amax) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < nel) ebad[i] = 0;
  if (i < n) sing[i] = 0;
  if (i < PIVOT_STATS) stats[i] = i < 3 ? 0 : INT_MAX;
  if (i == 0) *amax = 0.0;
}

// pivot statistics of the factor: out[0] negative pivots, out[1] true-zero
// and out[2] reduced-to-zero pivots replaced, out[3..5] the first such
// pivot columns, out[6] the first flagged element (INT_MAX: none); k_begin's
// start values
__global__ void k_pivot_stats(int n, const double* __restrict__ dpiv, const int* __restrict__ sing, int nel,
                              const int* __restrict__ ebad, int* __restrict__ out) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    if (sing[c]) {
      atomicAdd(&out[sing[c]], 1);
      atomicMin(&out[3 + sing[c]], c);
    } else if (dpiv[c] < 0.0) {
      atomicAdd(&out[0], 1);
      atomicMin(&out[3], c);
    }
  }
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nel; e += gridDim.x * blockDim.x)
    if (ebad[e]) atomicMin(&out[6], e);
}

// The reduced matrices in the reference's layout (CMSTRS, GRAV), nd x nd and
// column-major: first the n2 boundary rows in DOF order (pos2, 1-based), then
// the ngen component modes, zeros up to nd.  SK from the Schur complement
// (lower triangle of the root front, ld n2; null: left zero) and K11, SM from
// M22, M12 (ngen x n2) and M11, G (nd x 3) from Ge (n2 x 3) and Gg (ngen x 3),
// the products row-major, of squares the lower triangle; the element mass
// total follows.
// One launch and one copy instead of up to eight copies, each waited for.
__global__ __launch_bounds__(256) void k_reduced(int nd, int n2, int ngen, const int* __restrict__ pos2,
                                                 const double* __restrict__ S22, ReducedParts q,
                                                 const double* __restrict__ mass, double* __restrict__ out) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x, nn = (int64_t)nd * nd;
  const bool has_mass = mass != nullptr;
  if (g < nn) {
    const int i = (int)(g % nd), j = (int)(g / nd);
    double k = 0.0, m = 0.0;
    if (i < n2 && j < n2) {
      const int a = pos2[i] - 1, b = pos2[j] - 1, lo = min(a, b), hi = max(a, b);
      if (S22) k = S22[hi + (int64_t)lo * n2];
      if (has_mass) m = q.M22[(int64_t)hi * n2 + lo];
    } else if (min(i, j) >= n2 && max(i, j) < n2 + ngen) {
      const int at = (max(i, j) - n2) * ngen + min(i, j) - n2;
      k = q.K11[at];
      if (has_mass) m = q.M11[at];
    } else if (max(i, j) < n2 + ngen && has_mass) {
      m = q.M12[(int64_t)(max(i, j) - n2) * n2 + pos2[min(i, j)] - 1];
    }
    out[g] = k;
    if (has_mass) out[nn + g] = m;
  }
  if (has_mass && g < 3 * nd) {
    const int i = (int)(g % nd), c = (int)(g / nd);
    out[2 * nn + g] = i < n2 ? q.Ge[(pos2[i] - 1) * 3 + c] : i < n2 + ngen ? q.Gg[(i - n2) * 3 + c] : 0.0;
  }
  if (has_mass && g == 0) out[2 * nn + 3 * nd] = *mass;
}

__global__ void k_fill(double* __restrict__ p, int64_t n, double v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

// ---------------------------------------------------------------- front values
// The part of a front that no extend-add writes is cleared before the original
// entries are scattered into it: its own columns (the first ncol, which hold
// every original entry of a front but the Schur front's), and all of it where
// the front has no children or is the Schur front.  Task: sn, a = first of 16
// columns, k0 = end of the own columns; rows from the column block down (only
// the lower triangle has a meaning).
// Bound by HBM writes.  Clearing the whole pool took 3.0 ms for the 45x41x43
// block, this 0.8 ms.
template <class T>
__global__ __launch_bounds__(256) void k_front_zero(const FTask* __restrict__ tasks, DevSym S, T* __restrict__ pool) {
  const FTask t = tasks[blockIdx.x];
  const int ld = S.nrow[t.sn], lane = threadIdx.x & 63;
  T* F = pool + S.foff[t.sn];
  for (int j = t.a + (threadIdx.x >> 6); j < min(t.a + 16, t.k0); j += 4) {
    T* col = F + (int64_t)j * ld;
#pragma unroll 4
    for (int i = t.a + lane; i < ld; i += 64) col[i] = (T)0;
  }
}

// Task: sn = parent front, a = first parent column of a 16-column block, k0 =
// end of the own columns (above); blockIdx.y takes 512 of its rows from
// column a down.  The front's entries are gathered: the workgroup finds, child
// after child, which child row and column lands on each of its rows and
// columns (b/kb index the (child, first, end) column ranges in xrange, found
// when the schedule was built; the rows by a search in the child's sorted
// parent positions), adds the child's entries in registers and stores the
// block once.  Only own columns are read, the others start at zero, so the
// update part of a front is neither cleared nor read and written once per
// child.  Children are added in list order.
// Bound by HBM: one read of the children's update matrices and one write of
// the front.  Scattering each child into a cleared front took 7.1 + 3.0 ms
// for the 45x41x43 block, this 4.6 + 0.8 (18 GB: 4.0 TB/s), for the 48x24x24
// block 1.5 + 0.6 and 1.1 + 0.2.
constexpr int XADD_ROWS = 512;

template <class T>
__global__ __launch_bounds__(256) void k_extend_add(const FTask* __restrict__ tasks, DevSym S,
                                                    const int* __restrict__ xrange, T* __restrict__ pool) {
  __shared__ int srow[2][XADD_ROWS], scol[2][16];
  const FTask t = tasks[xcd_ranges(blockIdx.x, gridDim.x)];
  const int sn = t.sn, ld = S.nrow[sn], own = t.k0, c0 = t.a, tid = threadIdx.x, lane = tid & 63;
  const int r0 = c0 + XADD_ROWS * blockIdx.y;
  if (r0 >= ld || (t.kb == 0 && c0 + 16 <= own)) return;
  T* P = pool + S.foff[sn];
  const int halves = ld - r0 > 256 ? 2 : 1;  // 256 rows each
  T acc[2][16];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int r = r0 + 256 * h + tid;
#pragma unroll
    for (int c = 0; c < 16; c++) acc[h][c] = (T)0;
    if (c0 < own && h < halves) {
      const T* p = P + min(r, ld - 1);
#pragma unroll
      for (int c = 0; c < 16; c++) acc[h][c] = p[(int64_t)min(c0 + c, own - 1) * ld];
#pragma unroll
      for (int c = 0; c < 16; c++) acc[h][c] = c0 + c < own ? acc[h][c] : (T)0;
    }
  }
  for (int q = 0; q < t.kb; q++) {
    const int* xr = xrange + 3 * (t.b + q);
    const int ch = xr[0], a = xr[1], b = xr[2];
    const int nc = S.ncol[ch], ldc = S.nrow[ch], nu = ldc - nc;
    const int* rel = S.rel + S.relptr[ch];
    int* row = srow[q & 1];
    int* col = scol[q & 1];
    // a buffer is free once every thread has passed the barrier after the
    // next child's maps were made
    row[tid] = -1;
    row[tid + 256] = -1;
    if (tid < 16) col[tid] = -1;
    // first child row at or past r0: 64 probes a round, every wave for itself
    int lo = a, hi = blockIdx.y == 0 ? a : nu;
    while (lo < hi) {
      const int step = (hi - lo + 63) >> 6, at = lo + lane * step;
      const int less = __popcll(__ballot(at < hi && rel[min(at, hi - 1)] < r0));
      if (less == 0) break;
      hi = min(hi, lo + less * step);
      lo += (less - 1) * step + 1;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int i = lo + 256 * h + tid;
      const int p = rel[min(i, nu - 1)] - r0;
      if (i < nu && p < XADD_ROWS) row[p] = i;
    }
    if (tid < b - a) col[rel[a + tid] - c0] = a + tid;
    __syncthreads();
    const T* C = pool + S.foff[ch] + (int64_t)nc * ldc + nc;
    int jj[16];
#pragma unroll
    for (int c = 0; c < 16; c++) jj[c] = __builtin_amdgcn_readfirstlane(col[c]);
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int i = row[256 * h + tid];
      if (h >= halves || !__any(i >= 0)) continue;
      const T* src = C + max(i, a);  // unmatched rows and columns read another entry and drop it
      T v[16];
#pragma unroll
      for (int c = 0; c < 16; c++) v[c] = src[(int64_t)max(jj[c], a) * ldc];
#pragma unroll
      for (int c = 0; c < 16; c++) acc[h][c] = jj[c] >= 0 && i >= jj[c] ? acc[h][c] + v[c] : acc[h][c];
    }
  }
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int r = r0 + 256 * h + tid;
    if (r >= ld) continue;
#pragma unroll
    for (int c = 0; c < 16; c++)
      if (r >= c0 + c) P[r + (int64_t)(c0 + c) * ld] = acc[h][c];
  }
}

// ---------------------------------------------------------------- MFMA tile
// The 16x16x4 MFMA of the storage type (v_mfma_f64_16x16x4f64 for the FP64
// factor, v_mfma_f32_16x16x4f32 for the mixed-precision one).  The first
// operand takes the columns of a result tile and the second its rows, so for a
// fixed register consecutive lanes hold consecutive rows (coalesced stores into
// column-major fronts).  The two instructions place the 16x16 result
// differently: D[p][q] sits in lane q + 16*(p % 4), register p / 4 for FP64
// and in lane q + 16*(p / 4), register p % 4 for FP32.  Result register r: row
// lane & 15, column MF<T>::col(lane >> 4, r).
using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

template <class T> struct MF;
template <> struct MF<double> {
  using acc = f64x4;
  static __device__ __forceinline__ acc op(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int col(int lk, int r) { return lk + 4 * r; }
};
template <> struct MF<float> {
  using acc = f32x4;
  static __device__ __forceinline__ acc op(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int col(int lk, int r) { return 4 * lk + r; }
};

template <class A>
__device__ __forceinline__ void zero_acc(A (&acc)[2][2]) {
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++) acc[x][y] = A{};
}

// ---------------------------------------------------------------- panel
// a/d from r = recip64(d): the product corrected by its own residual (the
// quotient's rounding), three dependent operations instead of a division's
// scaling sequence.
__device__ __forceinline__ double quot64(double a, double d, double r) {
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-d, q, a), r, q);
}

// a/d in the storage type
__device__ __forceinline__ double div_pivot(double a, double d) { return quot64(a, d, recip64(d)); }
__device__ __forceinline__ float div_pivot(float a, double d) { return a / (float)d; }

// k_diag task: sn, k0 = first panel column.  Blocked LDL^T of the kb x kb
// (kb <= 64) diagonal block in LDS by four waves, in 16-column steps:
// (1) wave 0 factors the 16-column panel over all rows below its top, lane i
// holding row i in registers with readlane broadcasts, so L11, D1 and L21
// come out of one sweep; identity rows in the lanes that the panel leaves
// free turn into X11 = L11^-1 in the same sweep; (2) the tiles of the next
// panel's columns take A22 -= (L21 D1) L21^T on FP64 MFMA, one 16 x 16 tile
// per wave.  While wave 0 sweeps the next panel, waves 1-3 update the
// trailing tiles past it and form the off-diagonal tiles of X = L^-1,
// X_ij = -X_ii T_ij with T_ij = sum_{k=j}^{i-1} L_ik X_kj (wave j + 1 owns
// tile column j), so the chain of 64 pivots only waits for the sweeps and
// one tile each.  D goes to the pivot array, X into the diagonal tile of the
// pivot-block inverse pool.  The arithmetic is FP64 for both storage types
// (the FP32 factor of the mixed-precision path keeps its diagonal blocks'
// factorisation in FP64 and rounds only the stored result).  Rows beyond kb
// are carried as identity rows.
// Bound by the dependent chain over the pivots (a reciprocal, a quotient and
// a broadcast each): it sets the pace of every panel of the top separators.
// 64 pivots take about 25,000 cycles in one workgroup, nearly half of them in
// the four sweeps (2800 each, issue bound: 15 broadcasts by two readlanes and a
// product per pivot), most of the others in loads, stores and the panels' way to
// and from LDS.  A
// k_diag_trsm launch of the 117 x 109 plate takes 14.7 us (18.2 with LDS reads
// and stores under conditions, one wait each, and selects in the sweep that
// kept the unread upper entries; 37-39 with 16-row sweeps, a division per pivot
// and L21 through X11).
//
// diag_block: that factorisation in LDS; sA holds L below its unit diagonal,
// sD = D, sX = L^-1 with zeros above it, all in FP64 (sA on and above the
// diagonal holds left-overs).
template <class T>
__device__ __forceinline__ void diag_block(const T* __restrict__ F, int ld, int k0, int kb, double (&sA)[64][65],
                                           double (&sX)[64][65], double (&sD)[64], double (&sT)[4][16][17],
                                           const DevSym& S, int colbase) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  // singular-pivot test: |a_jj| of the block's columns, lane j of wave 0
  // holding column j, read once here
  const double amax = wv == 0 ? *S.amax : 0.0;
  const double adv = (wv == 0 && lane < kb) ? fabs(S.adiag[colbase + lane]) : 0.0;
  {
    // every load from inside the front and unconditional, the entries
    // outside the block replaced afterwards: a load under a condition waits
    // for the one before it
    const T* row = F + (int64_t)k0 * (ld + 1) + min(lane, kb - 1);
    T v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = row[(int64_t)min(wv + 4 * q, kb - 1) * ld];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int m = wv + 4 * q;
      sA[lane][m] = (lane < kb && m <= lane) ? (double)v[q] : (lane == m ? 1.0 : 0.0);
      sX[lane][m] = 0.0;
    }
  }
  __syncthreads();
  const int nsb = (kb + 15) >> 4;
  auto wave_fence = [&]() {  // this wave's LDS writes are visible to its own reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // A(ti, tj) -= (L(ti, p) D_p) L(tj, p)^T, 16 x 16 tiles, lower entries
  auto update_tile = [&](int ti, int tj, int p) {
    // (all reads at once, and of whole tiles: nobody reads the entries above
    // the diagonal)
    double a[4], b[4], c[4];
    double* out = &sA[16 * ti + lr][16 * tj + lk];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int m = 16 * p + 4 * q + lk;
      a[q] = sA[16 * tj + lr][m];
      b[q] = sA[16 * ti + lr][m] * sD[m];
      c[q] = out[4 * q];
    }
    f64x4 acc = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; q++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[q], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; r++) out[4 * r] = c[r] - acc[r];
  };
  // X_00 = L_00^-1 where the sweep had no free lanes: lane c < 16 solves
  // column c against the uniformly read L
  auto invert_tile0 = [&]() {
    if (lane < 16) {
      double x[16];
#pragma unroll
      for (int m = 0; m < 16; m++) x[m] = m == lane ? 1.0 : 0.0;
#pragma unroll
      for (int k = 0; k < 15; k++)
#pragma unroll
        for (int i = k + 1; i < 16; i++) x[i] = __builtin_fma(-sA[i][k], x[k], x[i]);
#pragma unroll
      for (int m = 0; m < 16; m++) sX[m][lane] = x[m];
    }
  };
  // T_ij into this wave's sT, then X_ij = -X_ii T_ij
  auto sum_tile = [&](int i, int j) {
    f64x4 acc = f64x4{0.0, 0.0, 0.0, 0.0};
    for (int kt = j; kt < i; kt++)
#pragma unroll
      for (int m0 = 0; m0 < 16; m0 += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sX[16 * kt + m0 + lk][16 * j + lr],
                                                   sA[16 * i + lr][16 * kt + m0 + lk], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; r++) sT[wv][lr][lk + 4 * r] = acc[r];
    wave_fence();
  };
  auto finish_tile = [&](int i, int j) {
    f64x4 acc = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m0 = 0; m0 < 16; m0 += 4)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sT[wv][m0 + lk][lr], sX[16 * i + lr][16 * i + m0 + lk], acc, 0, 0,
                                                 0);
#pragma unroll
    for (int r = 0; r < 4; r++) sX[16 * i + lr][16 * j + lk + 4 * r] = -acc[r];
    wave_fence();
  };
  for (int p = 0; p < nsb; p++) {
    const int c0 = 16 * p, used = 16 * (nsb - p);  // lanes that hold panel rows
    if (wv == 0) {
      // lane i holds row c0 + i of the panel; the sixteen lanes after the
      // panel's rows (when there are any) the rows of the identity
      const int row = min(c0 + lane, 63), unit = lane - used;
      double a[16], u[16];  // u: column j before its division by the pivot
      double d0;            // lane j: pivot c0 + j
      const double ac = __shfl(adv, (c0 + lane) & 63), thr = S.tolf * ac, rep = ac != 0.0 ? ac : amax;
      // TEST: a pivot below the limit is replaced (rare; the first pass only
      // detects it, as a select in the chain would slow every pivot)
      auto sweep = [&](auto test) {
        constexpr bool TEST = decltype(test)::value;
#pragma unroll
        for (int m = 0; m < 16; m++) u[m] = sA[row][c0 + m];
#pragma unroll
        for (int m = 0; m < 16; m++) a[m] = unit < 0 ? u[m] : (unit == m ? 1.0 : 0.0);
        auto pivot = [&](double v, int j) { return lane_bcast(TEST ? (fabs(v) > thr ? v : rep) : v, j); };
        d0 = a[0];
        double dj = pivot(a[0], 0), rj = recip64(dj);
#pragma unroll
        for (int j = 0; j < 16; j++) {
          u[j] = a[j];
          // the broadcasts of column j beside its quotient, then the next
          // pivot and its reciprocal beside the column updates
          double ub[16];
#pragma unroll
          for (int m = j + 1; m < 16; m++) ub[m] = lane_bcast(u[j], m);
          const double l = quot64(u[j], dj, rj);
          a[j] = l;  // (on and above the diagonal as well, where nobody reads it)
          if (j == 15) break;
          __builtin_amdgcn_sched_barrier(0);
          a[j + 1] = __builtin_fma(-l, ub[j + 1], a[j + 1]);
          d0 = lane == j + 1 ? a[j + 1] : d0;
          dj = pivot(a[j + 1], j + 1);
          rj = recip64(dj);
#pragma unroll
          for (int m = j + 2; m < 16; m++) a[m] = __builtin_fma(-l, ub[m], a[m]);
          __builtin_amdgcn_sched_barrier(0);  // the broadcasts stay in their step (few scalar registers)
        }
      };
      sweep(std::false_type{});
      const bool bad = lane < 16 && c0 + lane < kb && !(fabs(d0) > thr);
      if (__any(bad)) {
        sweep(std::true_type{});
        // column flags of the replaced pivots: 1 a true zero, 2 reduced to near zero
        if (lane < 16 && c0 + lane < kb && !(fabs(d0) > thr))
          S.sing[colbase + c0 + lane] = ac == 0.0 || fabs(d0) <= 1.0e3 * 2.220446049250313e-16 * ac ? 1 : 2;
      }
      if (unit < 0) {
        if (lane < 16) sD[c0 + lane] = fabs(d0) > thr ? d0 : rep;
#pragma unroll
        for (int m = 0; m < 16; m++) sA[row][c0 + m] = a[m];
      } else if (unit < 16) {
#pragma unroll
        for (int m = 0; m < 16; m++) sX[c0 + m][c0 + unit] = u[m];
      }
    } else if (p > 0) {
      // the work that the previous panel left: its row of X, T of this row if
      // it is the last, the trailing tiles (ti, tj), p < tj <= ti
      const int j = wv - 1, nt = nsb - p - 1;
      if (p == 1 && nsb == 4 && wv == 1) {
        invert_tile0();
        wave_fence();
      }
      if (j < p - 1) {
        sum_tile(p - 1, j);
        finish_tile(p - 1, j);
      }
      if (p == nsb - 1 && j < p) sum_tile(p, j);
      for (int q = (wv == 1 ? 2 : wv - 2); q < nt * (nt + 1) / 2; q += 3) {
        const int ti = q == 0 ? 0 : (q < 3 ? 1 : 2), tj = q - ti * (ti + 1) / 2;
        update_tile(p + 1 + ti, p + 1 + tj, p - 1);
      }
    }
    __syncthreads();
    if (p + 1 < nsb) {
      if (p + 1 + wv < nsb) update_tile(p + 1 + wv, p + 1, p);
      __syncthreads();
    }
  }
  if (wv > 0 && wv < nsb) finish_tile(nsb - 1, wv - 1);
  __syncthreads();
}

// L_r = F_r L_kk^-T D^-1 for a 64-row tile at row R0: sF the rows, sL =
// L_kk^-1 (lower, zeros above), C the panel's first column, d(j) its pivots
// (j < kb), read ahead of the products.  Wave w takes rows 16 w .. 16 w + 15;
// column tile y only sums over the column tiles m <= y, 40 MFMA steps a wave
// instead of 64.
template <class T, class D>
__device__ __forceinline__ void trsm_product(const T (*sF)[65], const T (*sL)[65], T* __restrict__ C, int ld, int R0,
                                             int kb, D d) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4, nsb = (kb + 15) >> 4;
  double dv[4][4];
#pragma unroll
  for (int y = 0; y < 4; y++)
#pragma unroll
    for (int r = 0; r < 4; r++) dv[y][r] = d(min(16 * y + MF<T>::col(lk, r), kb - 1));
  typename MF<T>::acc acc[4];
#pragma unroll
  for (int y = 0; y < 4; y++) acc[y] = typename MF<T>::acc{};
#pragma unroll
  for (int mt = 0; mt < 4; mt++) {
    if (mt >= nsb) break;
#pragma unroll
    for (int m0 = 0; m0 < 16; m0 += 4) {
      const int m = 16 * mt + m0 + lk;
      const T aa = sF[16 * wv + lr][m];
#pragma unroll
      for (int y = mt; y < 4; y++) acc[y] = MF<T>::op(sL[16 * y + lr][m], aa, acc[y]);
    }
  }
  const int i = R0 + 16 * wv + lr;
  if (i >= ld) return;
#pragma unroll
  for (int y = 0; y < 4; y++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int j = 16 * y + MF<T>::col(lk, r);
      if (j < kb) C[(int64_t)j * ld + i] = div_pivot(acc[y][r], dv[y][r]);
    }
}

// X = L^-1 into the diagonal tile of the pivot-block inverse pool and D into
// the pivot array.  The front's diagonal block itself is left alone (later kernels read D from the
// pivot array, the solves L^-1 from the inverse pool), so that other
// workgroups of the same launch can still read it.
template <class T>
__device__ __forceinline__ void diag_store(T* __restrict__ Xg, double* __restrict__ dpiv, int xld, int k0, int kb,
                                           int col0, const double (&sD)[64], const double (&sX)[64][65]) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid < kb) dpiv[col0 + k0 + tid] = sD[tid];
  double x[16];
#pragma unroll
  for (int q = 0; q < 16; q++) x[q] = sX[lane][wv + 4 * q];
  T* out = Xg + (int64_t)k0 * (xld + 1) + lane;
#pragma unroll
  for (int q = 0; q < 16; q++)
    if (lane < kb && wv + 4 * q < kb) out[(int64_t)(wv + 4 * q) * xld] = (T)x[q];
}

template <class T>
__global__ __launch_bounds__(256) void k_diag(const FTask* __restrict__ tasks, DevSym S,
                                              T* __restrict__ pool, const int64_t* __restrict__ ioff,
                                              T* __restrict__ ipool) {
  __shared__ double sA[64][65], sX[64][65], sD[64], sT[4][16][17];
  const FTask t = tasks[blockIdx.x];
  const int sn = t.sn, k0 = t.k0, ld = S.nrow[sn], nc = S.ncol[sn];
  const int kb = min(64, nc - k0);
  T* F = pool + S.foff[sn];
  T* Xg = ipool + ioff[sn];
  diag_block<T>(F, ld, k0, kb, sA, sX, sD, sT, S, S.col0[sn] + k0);
  diag_store<T>(Xg, S.dpiv, S.ild[sn], k0, kb, S.col0[sn], sD, sX);
}

// Diagonal block and triangular solve in one launch, for panels with few
// row tiles below the diagonal block (the upper levels of the tree, where a
// separate diagonal-block launch would run on a handful of CUs).  Task: sn,
// a = row tile (-1: none below), k0 = panel.  Every workgroup factors the
// diagonal block in LDS (the same FP64 arithmetic as k_diag, so the same
// bits); the one with a <= 0 stores it.  The row tile then takes
// L_r = F_r L_kk^{-T} D^{-1} with the factor values rounded to the storage
// type, exactly as k_trsm reads them back from memory.  The row tile's
// loads are issued before the factorisation.
template <class T>
__global__ __launch_bounds__(256) void k_diag_trsm(const FTask* __restrict__ tasks, DevSym S,
                                                   T* __restrict__ pool, const int64_t* __restrict__ ioff,
                                                   T* __restrict__ ipool) {
  __shared__ double sA[64][65], sX[64][65], sD[64], sT[4][16][17];
  const FTask t = tasks[xcd_ranges(blockIdx.x, gridDim.x)];
  const int sn = t.sn, k0 = t.k0, ld = S.nrow[sn], nc = S.ncol[sn];
  const int kb = min(64, nc - k0);
  T* F = pool + S.foff[sn];
  T* Xg = ipool + ioff[sn];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int R0 = k0 + kb + 64 * max(t.a, 0);
  T ra[16];
  if (t.a >= 0) {
    // in-front addresses (rows past the front and columns past the panel
    // repeat the last one; their products are not stored or meet a zero)
    const T* row = F + (int64_t)k0 * ld + min(R0 + lane, ld - 1);
#pragma unroll
    for (int q = 0; q < 16; q++) ra[q] = row[(int64_t)min(wv + 4 * q, kb - 1) * ld];
  }
  diag_block<T>(F, ld, k0, kb, sA, sX, sD, sT, S, S.col0[sn] + k0);
  if (t.a < 0) {
    diag_store<T>(Xg, S.dpiv, S.ild[sn], k0, kb, S.col0[sn], sD, sX);
    return;
  }
  // operand tiles in the storage type: the row tile in sA's space (every
  // read of sA is behind diag_block's last barrier), L^-1 in sX itself or,
  // rounded, behind the row tile
  T(*sF)[65] = reinterpret_cast<T(*)[65]>(&sA[0][0]);
  constexpr bool in_place = std::is_same<T, double>::value;
  T(*sL)[65] = in_place ? reinterpret_cast<T(*)[65]>(&sX[0][0]) : sF + 64;
#pragma unroll
  for (int q = 0; q < 16; q++) {
    sF[lane][wv + 4 * q] = wv + 4 * q < kb ? ra[q] : (T)0;
    if (!in_place) sL[lane][wv + 4 * q] = (T)sX[lane][wv + 4 * q];
  }
  __syncthreads();
  trsm_product<T>(sF, sL, F + (int64_t)k0 * ld, ld, R0, kb, [&](int j) { return sD[j]; });
  if (t.a == 0) diag_store<T>(Xg, S.dpiv, S.ild[sn], k0, kb, S.col0[sn], sD, sX);
}

// k_trsm task: sn, a = 64-row tile below the diagonal block, k0 = panel.
// L_r = F_r L_kk^{-T} D^{-1}, as an FP64 MFMA product with the inverse of the
// diagonal block built by k_diag.
template <class T>
__global__ __launch_bounds__(256) void k_trsm(const FTask* __restrict__ tasks, DevSym S,
                                              T* __restrict__ pool, const int64_t* __restrict__ ioff,
                                              const T* __restrict__ ipool) {
  __shared__ T sA[64][65];
  __shared__ T sB[64][65];
  const FTask t = tasks[xcd_ranges(blockIdx.x, gridDim.x)];
  const int sn = t.sn, k0 = t.k0, ld = S.nrow[sn], nc = S.ncol[sn];
  const int kb = min(64, nc - k0);
  const int R0 = k0 + kb + 64 * t.a;
  T* F = pool + S.foff[sn];
  const T* Xg = ipool + ioff[sn];
  const int xld = S.ild[sn];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  {
    // unconditional in-bounds loads, as in k_diag_trsm; sB[j][m] = Linv_kk[j][m] (lower)
    const T* row = F + (int64_t)k0 * ld + min(R0 + lane, ld - 1);
    const T* xrow = Xg + (int64_t)k0 * (xld + 1) + min(lane, kb - 1);
    T ra[16], rb[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int m = min(wv + 4 * q, kb - 1);
      ra[q] = row[(int64_t)m * ld];
      rb[q] = xrow[(int64_t)m * xld];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int m = wv + 4 * q;
      sA[lane][m] = m < kb ? ra[q] : (T)0;
      sB[lane][m] = (lane < kb && m <= lane) ? rb[q] : (T)0;
    }
  }
  __syncthreads();
  const double* dp = S.dpiv + S.col0[sn] + k0;
  trsm_product<T>(sA, sB, F + (int64_t)k0 * ld, ld, R0, kb, [&](int j) { return dp[j]; });
}

// ---------------------------------------------------------------- update
// Task: sn, a = ti, b = tj (64x64 tiles of the trailing lower triangle),
// k0 = panel, kb = panel width (<= 256), je = column limit; blockIdx.y the
// quadrant of the tile where a launch has four.  F[I,J] -= (L_I D) L_J^T over
// the panel.  A wave holds 16 XA x 16 YB of the tile in its MFMA accumulators
// and reads both operands straight from the panel, eight columns ahead of
// their products: a 16x16x4 FP64 step keeps the matrix core for 64 cycles, so
// the first-level cache feeds it without staging, barriers or staging
// arithmetic.  FP64: the accumulators start from the tile's current values and
// the J operand is scaled by -D, so the chain forms F - sum (L_I D) L_J^T and
// the tile is only stored at the end.  FP32 (mixed precision) sums the products
// from zero and subtracts them from the tile at the end: accumulating onto the
// tile through the FP32 MFMA left the factor too inexact for the FP64
// refinement of a thin 200x200 plate to converge.
// Bound by the matrix cores and by the rate of the first-level cache, which
// takes a quarter of a line a lane group: 16-byte loads of row pairs need half
// its cycles.  At 256 columns a panel two fronts of 6000 rows take 50 TFLOP/s
// and 16 of 1500 rows 51 (8-byte loads 43 and 44; waves of 64x64 46 and 40; at
// 128 columns, staged through LDS, 37 and 36); three or four chunks in flight
// and scalar address bases make no difference.  One front of 1900 rows has
// too few 64x32 waves (17 TFLOP/s, four waves of 32x32 24): the wide waves
// where a launch has UPD_WIDE or more tiles, else the four.  A tile of 256
// columns keeps the matrix cores of its CU for 7 us, so up to UPD_NARROW
// tiles, half as many as CUs, go as four workgroups of 32 x 32 each: 7 us a
// launch; 17x13x11 block 291 -> 230 us in all, 117x109 plate 671 -> 613 (limit
// 256: 237, 630; 512: 242, 659).
constexpr int UPD_WIDE = 2048, UPD_NARROW = 128;

template <int XA, int YB, class T>
__global__ __launch_bounds__(XA == 4 ? 128 : 256, XA == 4 ? 3 : 4) void k_update(const FTask* __restrict__ tasks, DevSym S,
                                                                T* __restrict__ pool) {
  constexpr int CH = 8, ST = CH / 4;
  const FTask t = tasks[xcd_ranges(blockIdx.x, gridDim.x)];
  const int sn = t.sn, k0 = t.k0, ld = S.nrow[sn], kb = t.kb;
  T* F = pool + S.foff[sn];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int quad = blockIdx.y;  // 0 of 1, or the quadrant of the tile
  const int I0 = k0 + kb + 64 * t.a + 32 * (quad >> 1) + 16 * XA * (wv >> 1);
  const int J0 = k0 + kb + 64 * t.b + 32 * (quad & 1) + 16 * YB * (wv & 1);
  const int je = t.je > 0 ? t.je : ld;
  if (I0 >= ld || J0 >= je || J0 >= I0 + 16 * XA) return;  // nothing of this part is stored
  // Rows go to the lanes in pairs where a wave has 32 of them: lane lr takes
  // rows 2 lr and 2 lr + 1, which are row lr of two MFMA tiles, by one 16-byte
  // load.  Rows past the front repeat its last one (and the entry behind it)
  // and are not stored.
  constexpr int VI = XA > 1 ? 2 : 1, VJ = YB > 1 ? 2 : 1;
  typedef T veci __attribute__((ext_vector_type(VI), aligned(sizeof(T))));
  typedef T vecj __attribute__((ext_vector_type(VJ), aligned(sizeof(T))));
  auto row_i = [&](int x) { return I0 + 16 * VI * x + VI * lr; };  // first row of lane's group x
  const T* base = F + (int64_t)(k0 + lk) * ld;
  const T *Ip[XA / VI], *Jp[YB / VJ];
#pragma unroll
  for (int x = 0; x < XA / VI; x++) Ip[x] = base + min(row_i(x), ld - 1);
#pragma unroll
  for (int y = 0; y < YB / VJ; y++) Jp[y] = base + min(J0 + 16 * VJ * y + VJ * lr, ld - 1);
  const double* Dp = S.dpiv + S.col0[sn] + k0;
  struct Stage {
    veci a[ST][XA / VI];
    vecj b[ST][YB / VJ];
    T d[ST];
  };
  // the next whole chunk, the pointers moving on (an address product per
  // load costs as much as the matrix step: 23 TFLOP/s)
  const int64_t step = (int64_t)4 * ld;
  const double* Dq = Dp + lk;
  auto load = [&](Stage& g) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
#pragma unroll
      for (int x = 0; x < XA / VI; x++) g.a[s][x] = *(const veci*)(Ip[x] + s * step);
#pragma unroll
      for (int y = 0; y < YB / VJ; y++) g.b[s][y] = *(const vecj*)(Jp[y] + s * step);
      g.d[s] = (T)Dq[4 * s];
    }
#pragma unroll
    for (int x = 0; x < XA / VI; x++) Ip[x] += ST * step;
#pragma unroll
    for (int y = 0; y < YB / VJ; y++) Jp[y] += ST * step;
    Dq += CH;
  };
  const int kf = kb & ~(2 * CH - 1);
  // a chunk from column c on, after the whole pairs of chunks; the columns
  // past the panel repeat the last one with a zero pivot
  auto load_tail = [&](int c, Stage& g) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const int k = c + 4 * s + lk, kc = min(k, kb - 1);
      const int64_t o = (int64_t)(kc - kf - lk) * ld;
#pragma unroll
      for (int x = 0; x < XA / VI; x++) g.a[s][x] = *(const veci*)(Ip[x] + o);
#pragma unroll
      for (int y = 0; y < YB / VJ; y++) g.b[s][y] = *(const vecj*)(Jp[y] + o);
      const T d = (T)Dp[kc];
      g.d[s] = k < kb ? d : (T)0;
    }
  };
  constexpr bool seed = std::is_same<T, double>::value;
  typename MF<T>::acc acc[XA][YB];
  auto multiply = [&](const Stage& g) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      T b[YB];
#pragma unroll
      for (int y = 0; y < YB; y++) {
        const T v = g.b[s][y / VJ][y % VJ] * g.d[s];
        b[y] = seed ? -v : v;
      }
#pragma unroll
      for (int x = 0; x < XA; x++)
#pragma unroll
        for (int y = 0; y < YB; y++) acc[x][y] = MF<T>::op(b[y], g.a[s][x / VI][x % VI], acc[x][y]);
    }
  };
  // column of the accumulators' entry r
  auto col_j = [&](int y, int r) { return J0 + 16 * VJ * (y / VJ) + VJ * MF<T>::col(lk, r) + y % VJ; };
  Stage g0, g1;
  if (kf > 0) load(g0);
#pragma unroll
  for (int x = 0; x < XA / VI; x++)
#pragma unroll
    for (int y = 0; y < YB; y++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        veci v{};
        if (seed) v = *(const veci*)(F + min(row_i(x), ld - 1) + (int64_t)min(col_j(y, r), ld - 1) * ld);
#pragma unroll
        for (int m = 0; m < VI; m++) acc[VI * x + m][y][r] = v[m];
      }
  // (no load under a condition in here: where the paths join, the compiler
  // waits for all that either may have in flight)
  for (int c = 2 * CH; c < kf; c += 2 * CH) {
    load(g1);
    multiply(g0);
    load(g0);
    multiply(g1);
  }
  if (kf > 0) {
    load(g1);
    multiply(g0);
    multiply(g1);
  }
  for (int c = kf; c < kb; c += CH) {
    load_tail(c, g0);
    multiply(g0);
  }
#pragma unroll
  for (int x = 0; x < XA / VI; x++)
#pragma unroll
    for (int y = 0; y < YB; y++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = row_i(x), j = col_j(y, r);
        if (i + VI - 1 < j || i >= ld || j >= je) continue;
        T* out = F + (int64_t)i + (int64_t)j * ld;
        veci v;
#pragma unroll
        for (int m = 0; m < VI; m++) v[m] = acc[VI * x + m][y][r];
        if (i >= j && i + VI <= ld) {
          *(veci*)out = seed ? v : *(veci*)out - v;
        } else {
#pragma unroll
          for (int m = 0; m < VI; m++)
            if (i + m >= j && i + m < ld) out[m] = seed ? v[m] : out[m] - v[m];
        }
      }
}

// ---------------------------------------------------------------- inverse
// Explicit inverse X = L_PP^{-1} of the unit lower-triangular pivot block of
// every front, kept in its own pool (ioff[s], ncol x ncol column-major, lower
// triangle).  With it each triangular solve of a front is a GEMM, which turns
// the forward/backward passes of the block Lanczos and of the B computation
// into a few wide launches per tree level instead of a sequence of dependent
// 64-column substitutions.
//
// The diagonal 64-column tiles come from the diagonal blocks.  From blocks of
// 64 h columns pairs are joined, h = 1, 2, 4, ...:
//   [X11     ]
//   [X21  X22]   X21 = -X22 T,  T = L21 X11
// by two launches over all fronts at once, so a front of n tiles takes 2 log2 n
// dependent launches of whole tiles instead of up to 2 n.
// k_inv_mul task: sn, a = tile column j, b = tile row i, k0 = the pair's first
// column of X22, kb = 0: T_ij = sum_{j<=k<k0} L_ik X_kj, 1: X_ij = -sum_{k0<=k<=i}
// X_ik T_kj, je = the place of the pair's T in tmp (16-element units; column-
// major, its rows those of X22).  Operands as in k_panel, three chunks ahead of
// their products (a small launch is bound by the latency of its loads); chunks
// past the sum repeat its last column and meet zeros.
// Fronts of 5544 and 3000 columns (45x41x43 block): 14 launches of 170 us
// (tile by tile at growing distance from the diagonal, staged through LDS: 164
// launches, 4.65 ms); 117x109 plate 8 of 19 us (16 launches, 223 us).
template <class T>
__global__ __launch_bounds__(256) void k_inv_mul(const FTask* __restrict__ tasks, DevSym S, const T* __restrict__ pool,
                                                 const int64_t* __restrict__ ioff, T* ipool, T* tmp) {
  const FTask t = tasks[blockIdx.x];
  const int sn = t.sn, ld = S.nrow[sn], nc = S.ncol[sn], xld = S.ild[sn], m = t.k0;
  const int h = (m / 64) & -(m / 64), first = m - 64 * h, end = min(m + 64 * h, nc), lt = end - m;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int i0 = 64 * t.b + (wv >> 1) * 32, j0 = 64 * t.a + (wv & 1) * 32;
  if (i0 >= end) return;
  const T* F = pool + S.foff[sn];
  T* X = ipool + ioff[sn];
  T* P = tmp + (int64_t)16 * t.je;  // element (i, j) of T at i - m + (j - first) lt
  const bool fin = t.kb != 0;
  // the sum from column kb on, kn of it (X is zero above its diagonal)
  const int kb = fin ? m : j0, kn = fin ? min(i0 + 32, end) - m : m - j0, lda = fin ? xld : ld;
  const T* A = (fin ? X : F) + (int64_t)kb * lda;
  const T* B = fin ? P + (int64_t)(j0 - first) * lt : X + (int64_t)j0 * xld + kb;
  const int ldb = fin ? lt : xld;
  const T *Ar[2], *Bc[2];
#pragma unroll
  for (int x = 0; x < 2; x++) {
    Ar[x] = A + min(i0 + 16 * x + lr, end - 1);
    Bc[x] = B + (int64_t)(16 * x + lr) * ldb;
  }
  constexpr int VK = 16 / sizeof(T);
  typedef T vec __attribute__((ext_vector_type(VK), aligned(sizeof(T))));
  struct Stage {
    T a[4][2], b[4][2];
  };
  auto kof = [&](int kc, int s) { return kc + 4 * VK * (s / VK) + VK * lk + s % VK; };
  auto load = [&](int kc, Stage& g) {
#pragma unroll
    for (int x = 0; x < 2; x++) {
#pragma unroll
      for (int s = 0; s < 4; s += VK) {
        const vec v = *(const vec*)(Bc[x] + min(kof(kc, s), kn - 1));
#pragma unroll
        for (int q = 0; q < VK; q++) g.b[s + q][x] = v[q];
      }
#pragma unroll
      for (int s = 0; s < 4; s++) g.a[s][x] = Ar[x][(int64_t)min(kof(kc, s), kn - 1) * lda];
    }
  };
  typename MF<T>::acc acc[2][2];
  zero_acc(acc);
  auto multiply = [&](int kc, const Stage& g) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const bool in = kof(kc, s) < kn;
#pragma unroll
      for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++) acc[x][y] = MF<T>::op(in ? g.b[s][y] : (T)0, in ? g.a[s][x] : (T)0, acc[x][y]);
    }
  };
  Stage g0, g1, g2, g3;
  load(0, g0);
  load(16, g1);
  load(32, g2);
  for (int kc = 0; kc < kn; kc += 64) {
    load(kc + 48, g3);
    multiply(kc, g0);
    load(kc + 64, g0);
    multiply(kc + 16, g1);
    load(kc + 80, g1);
    multiply(kc + 32, g2);
    load(kc + 96, g2);
    multiply(kc + 48, g3);
  }
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = i0 + 16 * x + lr, j = j0 + 16 * y + MF<T>::col(lk, r);
        if (i >= end) continue;
        if (fin) X[i + (int64_t)j * xld] = -acc[x][y][r];
        else P[i - m + (int64_t)(j - first) * lt] = acc[x][y][r];
      }
}

// Y21 = -L21 L11^-1 of a fused front, below L11^-1 in its solve panel, after
// every inverse tile.  Task: sn, a = 64-column tile j, b = 64-row tile i of
// the update rows: Y_ij = -sum_{k >= 64 j} L_ik X_kj.  Each wave forms a 32 x
// 32 quarter with both operands straight from memory (rows of L contiguous;
// X along k: each lane takes the VK neighbouring k of 16 bytes, step m of a
// 4 VK-chunk multiplies k = VK (lane / 16) + m), one chunk ahead of its
// products.  Both storage types add in FP64, so that a mixed-precision panel is
// rounded once (with FP32 sums a reduction takes as long, 102.9 ms of a 200x200
// plate).  The tasks come with the longest sums first and are dealt out one by
// one: in contiguous ranges per XCD the first XCD got all long ones (45x41x43
// block 2236 -> 890 us, 117x109 plate 265 -> 131, 17x13x11 block 52 -> 38).
template <class T>
__global__ __launch_bounds__(256) void k_panel(const FTask* __restrict__ tasks, DevSym S, const T* __restrict__ pool,
                                               const int64_t* __restrict__ ioff, T* __restrict__ ipool) {
  const FTask t = tasks[blockIdx.x];
  const int sn = t.sn, ld = S.nrow[sn], nc = S.ncol[sn], nu = ld - nc;
  const T* F = pool + S.foff[sn] + nc;
  T* Z = ipool + ioff[sn];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int i0 = 64 * t.b + (wv >> 1) * 32, j0 = 64 * t.a + (wv & 1) * 32;
  if (i0 >= nu || j0 >= nc) return;
  const T *Fr[2], *Xc[2];
#pragma unroll
  for (int x = 0; x < 2; x++) {
    Fr[x] = F + min(i0 + 16 * x + lr, nu - 1);
    Xc[x] = Z + (int64_t)min(j0 + 16 * x + lr, nc - 1) * ld;
  }
  constexpr int VK = 16 / sizeof(T);
  typedef T vec __attribute__((ext_vector_type(VK), aligned(sizeof(T))));
  struct Stage {
    T a[4][2], b[4][2];
  };
  auto kof = [&](int kc, int s) { return kc + 4 * VK * (s / VK) + VK * lk + s % VK; };
  auto load = [&](int kc, Stage& g) {
#pragma unroll
    for (int x = 0; x < 2; x++) {
#pragma unroll
      for (int s = 0; s < 4; s += VK) {
        const vec v = *(const vec*)(Xc[x] + min(kof(kc, s), nc - 1));
#pragma unroll
        for (int m = 0; m < VK; m++) g.b[s + m][x] = v[m];
      }
#pragma unroll
      for (int s = 0; s < 4; s++) g.a[s][x] = Fr[x][(int64_t)min(kof(kc, s), nc - 1) * ld];
    }
  };
  MF<double>::acc acc[2][2];
  zero_acc(acc);
  auto multiply = [&](int kc, const Stage& g) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const bool in = kof(kc, s) < nc;
#pragma unroll
      for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++) acc[x][y] = MF<double>::op(in ? (double)g.b[s][y] : 0.0, in ? (double)g.a[s][x] : 0.0, acc[x][y]);
    }
  };
  Stage g0, g1;
  const int kb = 64 * t.a;
  load(kb, g0);
  for (int kc = kb; kc < nc; kc += 32) {
    if (kc + 16 < nc) load(kc + 16, g1);
    multiply(kc, g0);
    if (kc + 16 >= nc) break;
    if (kc + 32 < nc) load(kc + 32, g0);
    multiply(kc + 16, g1);
  }
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = i0 + 16 * x + lr, j = j0 + 16 * y + MF<double>::col(lk, r);
        if (i < nu && j < nc) Z[(int64_t)nc + i + (int64_t)j * ld] = (T)-acc[x][y][r];
      }
}

// ---------------------------------------------------------------- products
// Z = A X for the full symmetric CSR matrix A (perm space), X, Z row-major.
// The rows of a node are neighbours and share their column list (the CSR rows
// are built from the node neighbours), so a wave takes the rows of one node,
// RB at a time, and gathers each row of X once for all of them.  It brings 64
// entries of the list and their values into its own LDS by loads of
// neighbouring places, the next 64 under the products, and its groups of W
// lanes take every (64 / W)-th entry: a lane gathers VEC neighbouring columns,
// NC times W VEC apart.  The groups' sums are added at the end; blockIdx.y
// takes the next W VEC NC columns.
// Bound by the load instructions of the gather (values and indices read by
// each group from memory: 2.5 times the time).  48x24x24 block (7.0 million
// entries) by 16 columns 92 -> 39 us, 45x41x43 194 -> 94, 90x84 plate by 66
// 142 -> 62, where a thread had a row and four columns.
template <int W, int VEC, int RB, int NC>
__global__ __launch_bounds__(256) void k_spmm(int nnode, int nrhs, const int* __restrict__ nrow0,
                                              const int* __restrict__ rowptr, const int* __restrict__ colind,
                                              const double* __restrict__ val, const double* __restrict__ X, int ldx,
                                              double* __restrict__ Z, int ldz) {
  constexpr int P = 64 / W, U = NC * VEC >= 4 ? 2 : 4;  // groups; gathers in flight of each
  typedef double vec __attribute__((ext_vector_type(VEC), aligned(8)));
  __shared__ double sv[4][RB][64];
  __shared__ int sc[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, j = lane % W, ph = lane / W;
  const int node = 4 * xcd_ranges(blockIdx.x, gridDim.x) + wv;
  if (node >= nnode) return;
  const int r0 = nrow0[node], dn = nrow0[node + 1] - r0;
  const int kb = rowptr[r0], len = rowptr[r0 + 1] - kb;
  // VEC columns from col(c) on (VEC divides nrhs), past the last ones these again
  auto col = [&](int c) { return (int)blockIdx.y * W * VEC * NC + VEC * (j + W * c); };
  const double* xb[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) xb[c] = X + min(col(c), nrhs - VEC);
  for (int rb = 0; rb < dn; rb += RB) {
    double acc[RB][NC][VEC];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int m = 0; m < VEC; m++) acc[i][c][m] = 0.0;
    int ci;
    double cv[RB];
    // entries past the list repeat its last one with a zero value
    auto load = [&](int k0) {
      const int k = min(k0 + lane, len - 1);
      ci = colind[kb + k];
#pragma unroll
      for (int i = 0; i < RB; i++) cv[i] = val[(int64_t)kb + (int64_t)min(rb + i, dn - 1) * len + k];
    };
    load(0);
    for (int k0 = 0; k0 < len; k0 += 64) {
      __builtin_amdgcn_wave_barrier();  // this wave's LDS keeps its order
      sc[wv][lane] = ci;
#pragma unroll
      for (int i = 0; i < RB; i++) sv[wv][i][lane] = k0 + lane < len ? cv[i] : 0.0;
      __builtin_amdgcn_wave_barrier();
      if (k0 + 64 < len) load(k0 + 64);
      const int n = min(64, len - k0);
      for (int e0 = 0; e0 < n; e0 += P * U) {
        vec x[U][NC];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int64_t o = (int64_t)sc[wv][(e0 + u * P + ph) & 63] * ldx;
#pragma unroll
          for (int c = 0; c < NC; c++) x[u][c] = *(const vec*)(xb[c] + o);
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int i = 0; i < RB; i++) {
            const double v = sv[wv][i][(e0 + u * P + ph) & 63];
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
              for (int m = 0; m < VEC; m++) acc[i][c][m] = __builtin_fma(v, x[u][c][m], acc[i][c][m]);
          }
      }
    }
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int c = 0; c < NC; c++) {
        vec s;
#pragma unroll
        for (int m = 0; m < VEC; m++) {
          double t = acc[i][c][m];
#pragma unroll
          for (int off = W; off < 64; off <<= 1) t += __shfl_xor(t, off);
          s[m] = t;
        }
        if (rb + i < dn && ph == (i * NC + c) % P && col(c) < nrhs) *(vec*)(Z + (int64_t)(r0 + rb + i) * ldz + col(c)) = s;
      }
  }
}

// Z = diag(A) X where A has no other value (the lumped mass of the shell
// elements in the stiffness' pattern, without constraints), dpos the diagonal's
// places.  A zero of the diagonal gives a zero row.  One pass over X and Z:
// 117x109 plate by 384 columns 325 -> 85 us.
constexpr int DIAG_ROWS = 2048;  // entries of Z per workgroup, whole rows

__global__ __launch_bounds__(256) void k_diag_mm(int n, int nrhs, int rows, const int* __restrict__ dpos,
                                                 const double* __restrict__ val, const double* __restrict__ X, int ldx,
                                                 double* __restrict__ Z, int ldz) {
  const int r0 = blockIdx.x * rows, end = min(rows, n - r0) * nrhs;
#pragma unroll 4
  for (int e = threadIdx.x; e < end; e += 256) {
    const int r = r0 + e / nrhs, j = e % nrhs;
    const double v = val[dpos[r]], x = X[(int64_t)r * ldx + j];
    Z[(int64_t)r * ldz + j] = v != 0.0 ? v * x : 0.0;
  }
}

// Sign convention of the component modes: for column i of Phi (rows in
// permuted order, ld columns), the component of largest magnitude over the
// internal equations taken in equation order (q -> row p1[q]; the first
// maximum wins) is made positive.  Pass 1: workgroup g scans equations
// g*span .. with lane -> column (64 columns at a time) and wave -> every
// fourth equation, and leaves per column its (|v|, v, q) best; pass 2: one
// wave per column combines the workgroups' bests (larger |v|, then smaller
// q), so the choice does not depend on scheduling.
__global__ __launch_bounds__(256) void k_mode_signs_part(int n1, int span, const int* __restrict__ p1,
                                                         const double* __restrict__ Phi, int ld, int nev,
                                                         double* __restrict__ best) {
  __shared__ double sa[4][64], sv[4][64];
  __shared__ int sq[4][64];
  const int g = blockIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int q0 = g * span, q1 = min(n1, q0 + span);
  for (int j0 = 0; j0 < nev; j0 += 64) {
    const int i = j0 + lane;
    double ba = -1.0, bv = 0.0;
    int bq = INT_MAX;
    if (i < nev)
      for (int q = q0 + wv; q < q1; q += 4) {  // q ascends within a lane
        const double v = Phi[(int64_t)p1[q] * ld + i], a = fabs(v);
        if (a > ba) { ba = a; bv = v; bq = q; }
      }
    sa[wv][lane] = ba;
    sv[wv][lane] = bv;
    sq[wv][lane] = bq;
    __syncthreads();
    if (wv == 0 && i < nev) {
      for (int w = 1; w < 4; w++) {
        const double a2 = sa[w][lane];
        const int q2 = sq[w][lane];
        if (a2 > ba || (a2 == ba && q2 < bq)) { ba = a2; bv = sv[w][lane]; bq = q2; }
      }
      double* o = best + ((int64_t)g * nev + i) * 3;
      o[0] = ba;
      o[1] = bv;
      o[2] = (double)bq;
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(64) void k_mode_signs_fin(int ngroups, int nev, const double* __restrict__ best,
                                                       double* __restrict__ sign) {
  const int i = blockIdx.x, lane = threadIdx.x;
  double ba = -1.0, bv = 0.0, bq = 1e300;
  for (int g = lane; g < ngroups; g += 64) {
    const double* o = best + ((int64_t)g * nev + i) * 3;
    if (o[0] > ba || (o[0] == ba && o[2] < bq)) { ba = o[0]; bv = o[1]; bq = o[2]; }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double a2 = __shfl_xor(ba, off), v2 = __shfl_xor(bv, off), q2 = __shfl_xor(bq, off);
    if (a2 > ba || (a2 == ba && q2 < bq)) { ba = a2; bv = v2; bq = q2; }
  }
  if (lane == 0) sign[i] = bv < 0.0 ? -1.0 : 1.0;
}

__global__ void k_scale_cols(int64_t n, int nc, const double* __restrict__ sign, double* __restrict__ X) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g < n * nc) X[g] *= sign[g % nc];
}

// X[(ndof1 + b) * nrhs + b] = 1, all other entries 0 (the [B; I] identity rows)
__global__ void k_identity_rows(double* __restrict__ X, int64_t nrows, int nrhs, int ndof1) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nrows * nrhs) return;
  int64_t r = g / nrhs;
  int j = (int)(g % nrhs);
  X[g] = (r >= ndof1 && r - ndof1 == j) ? 1.0 : 0.0;
}

// Element mass EMASS of lhsINADD (inadd.f90:258-265): the x-translation mass
// u_x^T M_e u_x of each element's packed node-pair blocks (diagonal blocks
// once, off-diagonal blocks twice; entry (0,0) of a block couples the two
// nodes' x translations).  One lane per element of one type list.
__global__ void k_emass(int n, const int* __restrict__ elist, int nen, int d, const int64_t* __restrict__ eoff,
                        const double* __restrict__ Mp, double* __restrict__ emass) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int e = elist[t];
  const double* m = Mp + eoff[e];
  double s = 0.0;
  for (int a = 0; a < nen; a++)
    for (int b = 0; b <= a; b++) s += (a == b ? 1.0 : 2.0) * m[(int64_t)(a * (a + 1) / 2 + b) * d * d];
  emass[e] = s;
}

// out[0] = sum of x[0..n-1] by one workgroup in a fixed order (strided lane
// sums, then a tree), so the total is the same bits on every run
__global__ __launch_bounds__(256) void k_sum_fixed(int n, const double* __restrict__ x, double* __restrict__ out) {
  __shared__ double red[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += x[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// ---------------------------------------------------------------- Lanczos start block
// Deterministic pseudo-random values in (-1/2, 1/2) on the first n1 rows of
// the row-major neq x bs block, zeros below: entry g of the rows takes the
// (g + 1)-th output of the SplitMix64 sequence of the seed (Steele, Lea and
// Flood 2014), whose state is a plain multiple of the step, so every entry
// stands alone.  Made here because the host took 3 ms and its copy 1.5 ms
// for a 91,839 x 16 block, with the device idle (now 3 us).
__global__ void k_start_block(int64_t n, int64_t n1, uint64_t seed, double* __restrict__ W) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  uint64_t z = seed + (uint64_t)(g + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  W[g] = g < n1 ? (double)(z >> 11) * (1.0 / 9007199254740992.0) - 0.5 : 0.0;
}

// ---------------------------------------------------------------- mixed precision
// Symmetric diagonal equilibration of the stiffness matrix for the FP32
// factor: s[r] = 1/sqrt(K[r][r]) for every perm row r of the CSR matrix
// (1 for a non-positive diagonal, which the factorisation then reports).
__global__ void k_diag_scale(int n, const int* __restrict__ dpos, const double* __restrict__ val,
                             double* __restrict__ s) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const double d = val[dpos[r]];
  s[r] = d != 0.0 ? 1.0 / sqrt(fabs(d)) : 1.0;
}

// The equilibrated stiffness s_r K_rc s_c of every lower CSR entry into its
// FP32 front position (the FP64 factor takes the entries from k_assemble).
__global__ void k_front_scatter32(int n, const int* __restrict__ rowptr, const int* __restrict__ colind,
                                  const double* __restrict__ val, const double* __restrict__ s,
                                  const int64_t* __restrict__ fmap, float* __restrict__ pool) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  for (int k = rowptr[r]; k < rowptr[r + 1]; k++) {
    const int64_t f = fmap[k];
    if (f >= 0) pool[f] = (float)(s[r] * val[k] * s[colind[k]]);
  }
}

// Y[r][j] = X[r][j] rs[r] (rows 0..nrows-1) and, with cs, times cs[j]
// (row-major, nrhs columns; Y may be X)
__global__ void k_scale_rc(int64_t nrows, int nrhs, const double* __restrict__ rs, const double* __restrict__ cs,
                           const double* X, double* Y) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nrows * nrhs) return;
  const int64_t r = g / nrhs;
  const int j = (int)(g % nrhs);
  double v = X[g] * rs[r];
  if (cs) v *= cs[j];
  Y[g] = v;
}

// y[i] = 1 / x[i]
__global__ void k_recip(int n, const double* __restrict__ x, double* __restrict__ y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = 1.0 / x[i];
}

// Y = a X + b Y over the first n entries (Y not read when b = 0; X and Y may be
// the same array)
__global__ void k_axpby(int64_t n, double a, const double* X, double b, double* Y) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g < n) Y[g] = b == 0.0 ? a * X[g] : a * X[g] + b * Y[g];
}

// part[blk] = (sum x^2, sum y^2) over the block's slice of the first n
// entries; the host adds the blocks in order (deterministic norms)
__global__ __launch_bounds__(256) void k_sumsq2(int64_t n, const double* __restrict__ x,
                                                const double* __restrict__ y, double* __restrict__ part) {
  __shared__ double r0[256], r1[256];
  double a = 0.0, b = 0.0;
  const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
  const int64_t lo = (int64_t)blockIdx.x * chunk, hi = min(n, lo + chunk);
  for (int64_t i = lo + threadIdx.x; i < hi; i += 256) {
    a += x[i] * x[i];
    b += y[i] * y[i];
  }
  r0[threadIdx.x] = a;
  r1[threadIdx.x] = b;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      r0[threadIdx.x] += r0[threadIdx.x + w];
      r1[threadIdx.x] += r1[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r0[0];
    part[2 * blockIdx.x + 1] = r1[0];
  }
}

// Column dot products of up to three pairs (A_k, B_k) of row-major n x nr
// arrays: block b sums rows [b COLDOT_ROWS, (b+1) COLDOT_ROWS) of each column
// into part[(b * npair + k) * nr + c].  Its threads stand W = min(nr, 256)
// columns wide and as many rows high as fit, take every so many-th row and
// add their sums in row order through LDS; k_coldot_sum then adds the blocks
// in a fixed order (16 groups of them per column).  Bound by HBM: 45,000 rows
// by 66 columns, one to three pairs, 158 + 44 -> 16 + 9 us on average (one
// thread per column and 256 rows, one thread per column over all blocks).
__global__ __launch_bounds__(256) void k_coldot_part(int64_t n, int nr, int npair, const double* __restrict__ A0,
                                                     const double* __restrict__ B0, const double* __restrict__ A1,
                                                     const double* __restrict__ B1, const double* __restrict__ A2,
                                                     const double* __restrict__ B2, double* __restrict__ part) {
  __shared__ double red[3][256];
  const int W = min(nr, 256), H = 256 / W, tid = threadIdx.x, g = tid / W;
  const int64_t r0 = (int64_t)blockIdx.x * COLDOT_ROWS, r1 = min(n, r0 + COLDOT_ROWS);
  for (int c0 = 0; c0 < nr; c0 += W) {
    const int c = c0 + tid % W;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    if (g < H && c < nr) {
      if (npair == 3) {
#pragma unroll 4
        for (int64_t r = r0 + g; r < r1; r += H) {
          const int64_t o = r * nr + c;
          s0 += A0[o] * B0[o];
          s1 += A1[o] * B1[o];
          s2 += A2[o] * B2[o];
        }
      } else if (npair == 2) {
#pragma unroll 4
        for (int64_t r = r0 + g; r < r1; r += H) {
          const int64_t o = r * nr + c;
          s0 += A0[o] * B0[o];
          s1 += A1[o] * B1[o];
        }
      } else {
#pragma unroll 4
        for (int64_t r = r0 + g; r < r1; r += H) s0 += A0[r * nr + c] * B0[r * nr + c];
      }
    }
    red[0][tid] = s0;
    red[1][tid] = s1;
    red[2][tid] = s2;
    __syncthreads();
    if (tid < W && c < nr)
      for (int k = 0; k < npair; k++) {
        double s = red[k][tid];
        for (int h = 1; h < H; h++) s += red[k][h * W + tid];
        part[((int64_t)blockIdx.x * npair + k) * nr + c] = s;
      }
    __syncthreads();
  }
}

__global__ __launch_bounds__(1024) void k_coldot_sum(int nb, int n, const double* __restrict__ part,
                                                     double* __restrict__ out) {
  __shared__ double red[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, idx = blockIdx.x * 64 + lane;
  const double* p = part + min(idx, n - 1);
  double s = 0.0;
  int b = w;
  for (; b + 7 * 16 < nb; b += 8 * 16) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = p[(int64_t)(b + 16 * u) * n];
#pragma unroll
    for (int u = 0; u < 8; u++) s += v[u];
  }
  for (; b < nb; b += 16) s += p[(int64_t)b * n];
  red[w][lane] = s;
  __syncthreads();
  if (w > 0 || idx >= n) return;
#pragma unroll
  for (int k = 1; k < 16; k++) s += red[k][lane];
  out[idx] = s;
}

// Y[r][c] = a[c] X[r][c] + b[c] Y[r][c] over n rows of row-major n x nr
// arrays (a or b null: coefficient 1).
__global__ __launch_bounds__(256) void k_col_axpby(int64_t n, int nr, const double* __restrict__ a,
                                                   const double* __restrict__ X, const double* __restrict__ b,
                                                   double* __restrict__ Y) {
  const int64_t total = n * nr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int c = (int)(i % nr);
    const double ya = b ? b[c] * Y[i] : Y[i];
    Y[i] = (a ? a[c] * X[i] : X[i]) + ya;
  }
}

// ---------------------------------------------------------------- launchers
void launch_hex8(hipStream_t st, int nhex, const int* elist, const int* eptr, const int* enodes,
                 const double* xyz, const double* eprop, const int64_t* eoff, double* Kp, double* Mp,
                 int* ebad) {
  if (nhex > 0) k_hex8<<<nhex, 64, 0, st>>>(nhex, elist, eptr, enodes, xyz, eprop, eoff, Kp, Mp, ebad);
}
void launch_assemble(hipStream_t st, int64_t nnz, const int* cptr, const int* cidx, const double* ccoef,
                     const double* Kp, const double* Mp, double* Kv, double* Mv, const int64_t* fmap, double* pool) {
  if (nnz <= 0) return;
  if (ccoef) k_assemble<true><<<nblk(nnz, 256), 256, 0, st>>>(nnz, cptr, cidx, ccoef, Kp, Mp, Kv, Mv, fmap, pool);
  else k_assemble<false><<<nblk(nnz, 256), 256, 0, st>>>(nnz, cptr, cidx, ccoef, Kp, Mp, Kv, Mv, fmap, pool);
}
void launch_diag_extract(hipStream_t st, int n, const int* dpos, const double* val, const double* rs, double* adiag,
                         double* amax) {
  if (n > 0)
    k_diag_extract<<<std::min(256u, nblk(n, 256)), 256, 0, st>>>(n, dpos, val, rs, adiag,
                                                                 reinterpret_cast<unsigned long long*>(amax));
}
void launch_begin(hipStream_t st, int nel, int* ebad, int n, int* sing, int* stats, double* amax) {
  k_begin<<<nblk(std::max({nel, n, PIVOT_STATS}), 256), 256, 0, st>>>(nel, ebad, n, sing, stats, amax);
}
void launch_pivot_stats(hipStream_t st, int n, const double* dpiv, const int* sing, int nel, const int* ebad,
                        int* out) {
  const int most = std::max(n, nel);
  if (most > 0) k_pivot_stats<<<std::min(1024u, nblk(most, 256)), 256, 0, st>>>(n, dpiv, sing, nel, ebad, out);
}
void launch_reduced(hipStream_t st, int nd, int n2, int ngen, const int* pos2, const double* S22,
                    const ReducedParts& q, const double* mass, double* out) {
  const int64_t n = std::max((int64_t)nd * nd, (int64_t)3 * nd + 1);
  k_reduced<<<nblk(n, 256), 256, 0, st>>>(nd, n2, ngen, pos2, S22, q, mass, out);
}
void launch_fill(hipStream_t st, double* p, int64_t n, double v) {
  if (n > 0) k_fill<<<(unsigned)std::min<int64_t>(nblk(n, 256), 16384), 256, 0, st>>>(p, n, v);
}
#define FGPU_FACTOR_LAUNCHERS(T)                                                                          \
  void launch_front_zero(hipStream_t st, const FTask* t, int n, const DevSym& S, T* pool) {               \
    if (n > 0) k_front_zero<T><<<n, 256, 0, st>>>(t, S, pool);                                            \
  }                                                                                                       \
  void launch_extend_add(hipStream_t st, const FTask* t, int n, int rows, const DevSym& S,                \
                         const int* xrange, T* pool) {                                                    \
    if (n > 0) k_extend_add<T><<<dim3(n, nblk(rows, XADD_ROWS)), 256, 0, st>>>(t, S, xrange, pool);       \
  }                                                                                                       \
  void launch_diag(hipStream_t st, const FTask* t, int n, const DevSym& S, T* pool, const int64_t* ioff,  \
                   T* ipool) {                                                                            \
    if (n > 0) k_diag<T><<<n, 256, 0, st>>>(t, S, pool, ioff, ipool);                                     \
  }                                                                                                       \
  void launch_diag_trsm(hipStream_t st, const FTask* t, int n, const DevSym& S, T* pool,                  \
                        const int64_t* ioff, T* ipool) {                                                  \
    if (n > 0) k_diag_trsm<T><<<n, 256, 0, st>>>(t, S, pool, ioff, ipool);                                \
  }                                                                                                       \
  void launch_trsm(hipStream_t st, const FTask* t, int n, const DevSym& S, T* pool, const int64_t* ioff,  \
                   const T* ipool) {                                                                      \
    if (n > 0) k_trsm<T><<<n, 256, 0, st>>>(t, S, pool, ioff, ipool);                                     \
  }                                                                                                       \
  void launch_update(hipStream_t st, const FTask* t, int n, const DevSym& S, T* pool) {                   \
    if (n >= UPD_WIDE) k_update<4, 2, T><<<n, 128, 0, st>>>(t, S, pool);                                  \
    else if (n > UPD_NARROW) k_update<2, 2, T><<<n, 256, 0, st>>>(t, S, pool);                            \
    else if (n > 0) k_update<1, 1, T><<<dim3(n, 4), 256, 0, st>>>(t, S, pool);                            \
  }                                                                                                       \
  void launch_inv_mul(hipStream_t st, const FTask* t, int n, const DevSym& S, const T* pool,              \
                      const int64_t* ioff, T* ipool, T* tmp) {                                            \
    if (n > 0) k_inv_mul<T><<<n, 256, 0, st>>>(t, S, pool, ioff, ipool, tmp);                             \
  }                                                                                                       \
  void launch_panel(hipStream_t st, const FTask* t, int n, const DevSym& S, const T* pool,                \
                    const int64_t* ioff, T* ipool) {                                                      \
    if (n > 0) k_panel<T><<<n, 256, 0, st>>>(t, S, pool, ioff, ipool);                                    \
  }
FGPU_FACTOR_LAUNCHERS(double)
FGPU_FACTOR_LAUNCHERS(float)
#undef FGPU_FACTOR_LAUNCHERS
void launch_spmm(hipStream_t st, const NodeRows& nr, int nrhs, const int* rowptr, const int* colind, const double* val,
                 const double* X, int ldx, double* Z, int ldz) {
  if (nr.nnode <= 0 || nrhs <= 0) return;
  // columns in as even groups as tiles of 16 allow, up to 64 a wave, in pairs
  // where they are even; three rows at a time where most nodes have no more
  // (solids), else six
  const int groups = (nrhs + 63) / 64, nc = (nrhs + 16 * groups - 1) / (16 * groups);
  using std::integral_constant;
  auto go = [&](auto w, auto vec, auto rb, auto c) {
    constexpr int W = decltype(w)::value, VEC = decltype(vec)::value, NC = decltype(c)::value;
    k_spmm<W, VEC, decltype(rb)::value, NC><<<dim3(nblk(nr.nnode, 4), nblk(nrhs, W * VEC * NC)), 256, 0, st>>>(
        nr.nnode, nrhs, nr.row0, rowptr, colind, val, X, ldx, Z, ldz);
  };
  auto by_cols = [&](auto rb) {
    using W4 = integral_constant<int, 4>;
    using W8 = integral_constant<int, 8>;
    using W16 = integral_constant<int, 16>;
    using C1 = integral_constant<int, 1>;
    using C2 = integral_constant<int, 2>;
    if (nrhs <= 4) go(W4{}, C1{}, rb, C1{});
    else if (nrhs % 2) nc == 1 ? go(W16{}, C1{}, rb, C1{}) : go(W16{}, C1{}, rb, C2{});
    else if (nc == 1) go(W8{}, C2{}, rb, C1{});
    else if (nc == 2) go(W8{}, C2{}, rb, C2{});
    else if (nc == 3) go(W8{}, C2{}, rb, integral_constant<int, 3>{});
    else go(W8{}, C2{}, rb, integral_constant<int, 4>{});
  };
  if (2 * nr.nrow < 9 * nr.nnode) by_cols(integral_constant<int, 3>{});
  else by_cols(integral_constant<int, 6>{});
}
void launch_diag_mm(hipStream_t st, int n, int nrhs, const int* dpos, const double* val, const double* X, int ldx,
                    double* Z, int ldz) {
  const int rows = std::max(1, DIAG_ROWS / std::max(1, nrhs));
  if (n > 0 && nrhs > 0) k_diag_mm<<<nblk(n, rows), 256, 0, st>>>(n, nrhs, rows, dpos, val, X, ldx, Z, ldz);
}
void launch_mode_signs(hipStream_t st, int n1, const int* p1, double* Phi, int64_t nrows, int nev, double* sign) {
  if (nev <= 0) return;
  // sign[0 .. nev) is the result; the groups' bests follow it
  double* best = sign + nev;
  const int span = std::max(1, (n1 + MODE_SIGN_GROUPS - 1) / MODE_SIGN_GROUPS);
  const int ng = std::max(1, (n1 + span - 1) / span);
  k_mode_signs_part<<<ng, 256, 0, st>>>(n1, span, p1, Phi, nev, nev, best);
  k_mode_signs_fin<<<nev, 64, 0, st>>>(ng, nev, best, sign);
  if (nrows > 0) k_scale_cols<<<nblk(nrows * nev, 256), 256, 0, st>>>(nrows, nev, sign, Phi);
}
void launch_emass(hipStream_t st, int n, const int* elist, int nen, int d, const int64_t* eoff, const double* Mp,
                  double* emass) {
  if (n > 0) k_emass<<<nblk(n, 256), 256, 0, st>>>(n, elist, nen, d, eoff, Mp, emass);
}
void launch_sum_fixed(hipStream_t st, int n, const double* x, double* out) {
  k_sum_fixed<<<1, 256, 0, st>>>(n, x, out);
}
void launch_start_block(hipStream_t st, int neq, int n1, int bs, uint64_t seed, double* W) {
  const int64_t n = (int64_t)neq * bs;
  if (n > 0) k_start_block<<<nblk(n, 256), 256, 0, st>>>(n, (int64_t)n1 * bs, seed, W);
}
void launch_diag_scale(hipStream_t st, int n, const int* dpos, const double* val, double* s) {
  if (n > 0) k_diag_scale<<<nblk(n, 256), 256, 0, st>>>(n, dpos, val, s);
}
void launch_front_scatter32(hipStream_t st, int n, const int* rowptr, const int* colind, const double* val,
                            const double* s, const int64_t* fmap, float* pool) {
  if (n > 0) k_front_scatter32<<<nblk(n, 256), 256, 0, st>>>(n, rowptr, colind, val, s, fmap, pool);
}
void launch_scale_rc(hipStream_t st, int64_t nrows, int nrhs, const double* rs, const double* cs, const double* X,
                     double* Y) {
  if (nrows * nrhs > 0) k_scale_rc<<<nblk(nrows * nrhs, 256), 256, 0, st>>>(nrows, nrhs, rs, cs, X, Y);
}
void launch_recip(hipStream_t st, int n, const double* x, double* y) {
  if (n > 0) k_recip<<<nblk(n, 256), 256, 0, st>>>(n, x, y);
}
void launch_axpby(hipStream_t st, int64_t n, double a, const double* X, double b, double* Y) {
  if (n > 0) k_axpby<<<nblk(n, 256), 256, 0, st>>>(n, a, X, b, Y);
}
int coldot_blocks(int64_t n) { return (int)((n + COLDOT_ROWS - 1) / COLDOT_ROWS); }
void launch_coldots(hipStream_t st, int64_t n, int nr, int npair, const double* A0, const double* B0,
                    const double* A1, const double* B1, const double* A2, const double* B2, double* part,
                    double* out) {
  const int nb = coldot_blocks(n);
  if (nb > 0) k_coldot_part<<<nb, 256, 0, st>>>(n, nr, npair, A0, B0, A1, B1, A2, B2, part);
  k_coldot_sum<<<nblk((int64_t)npair * nr, 64), 1024, 0, st>>>(nb, npair * nr, part, out);
}
void launch_col_axpby(hipStream_t st, int64_t n, int nr, const double* a, const double* X, const double* b,
                      double* Y) {
  const int64_t total = n * nr;
  if (total > 0) k_col_axpby<<<(unsigned)std::min<int64_t>(nblk(total, 256), 8192), 256, 0, st>>>(n, nr, a, X, b, Y);
}
void launch_sumsq2(hipStream_t st, int64_t n, const double* x, const double* y, double* part) {
  k_sumsq2<<<SUMSQ_BLOCKS, 256, 0, st>>>(n, x, y, part);
}
void launch_identity_rows(hipStream_t st, double* X, int64_t nrows, int nrhs, int ndof1) {
  if (nrows * nrhs > 0) k_identity_rows<<<nblk(nrows * nrhs, 256), 256, 0, st>>>(X, nrows, nrhs, ndof1);
}

}  // namespace fgpu
