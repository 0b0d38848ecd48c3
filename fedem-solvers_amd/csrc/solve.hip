// Multi-RHS triangular solves with the multifrontal factor on gfx950.
//
// Multi-vectors are row-major (rows x nrhs).  Work buffer W holds, for front
// s, rows woff[s] .. woff[s]+nrow[s]-1.  The solve panel of a front holds
// X11 = L11^-1 (unit lower triangular, zeros above it in the diagonal tiles)
// and, in a fused level, Y21 = -L21 X11 below it, so that one product does a
// level's forward step and one its backward step:
//   forward   [v; du] = [X11; Y21] w_p,  y_p = D^-1 v,  w_u += du
//   backward  x_p = X11^T y_p + Y21^T x_u
// An unfused level (large fronts, where forming Y21 costs more than the
// launches it saves) multiplies by X11 and by L21 of the front in turn.
#include <algorithm>
#include "kern_device.hpp"

namespace fgpu {

// The tasks of a launch go to the XCDs by fours (xcd_fours): neighbours share
// source rows and the lines between their target rows.  Whole ranges per XCD
// gave one the short and another the long sums of a triangular block: the
// products of a Lanczos step of the 45x41x43 block 2074 -> 1950 us, 48x24x24
// 642 -> 610.

// Result v of target row r, right-hand side j of task t.  GM > 0: base is what
// the children add to a row of W, which the row itself does not hold.
template <int GM, class T>
__device__ __forceinline__ void mv_apply(const MvTask& t, int r, int j, double v, double base,
                                         const double* __restrict__ dpiv, double* W, double* V, double* Y, double* X,
                                         int nrhs) {
  double* w = W + (int64_t)(t.dst + r) * nrhs + j;
  switch (t.flags & MV_APPLY) {
    case MV_Y:
      if (t.dst2 >= 0) V[(int64_t)(t.dst2 + r) * nrhs + j] = v;
      Y[(int64_t)(t.dst + r) * nrhs + j] = v / (double)(T)dpiv[t.dst + r];
      break;
    case MV_SET: *w = v; break;
    case MV_NEG: *w = -v; break;
    case MV_ADD: *w = (GM ? base : *w) + v; break;
    case MV_SUB: *w = (GM ? base : *w) - v; break;
    case MV_X: X[(int64_t)(t.dst + r) * nrhs + j] = v; break;
    default:  // MV_YSUB
      *w = (Y ? Y[(int64_t)(t.dst2 + r) * nrhs + j] : 0.0) - v;
  }
}

// Sum of the K parts' 16 x 16 NT results in part order through LDS (red: KW
// x 16 x 17 values) and their application; acc[y][q] holds target row lr,
// right-hand side 16 y + lk + 4 q; base[y] belongs to row (thread / 16) mod 16,
// right-hand side 16 y + thread mod 16.
template <int NT, int KW, int GM, class T>
__device__ __forceinline__ void mv_combine(const MvTask& t, const f64x4 (&acc)[NT], const double (&base)[NT],
                                           double* red, const double* __restrict__ dpiv, double* W, double* V, double* Y,
                                           double* X, int nrhs) {
  const int lane = threadIdx.x & 63, kw = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int y = 0; y < NT; y++) {
    if (y > 0) __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++) red[kw * 272 + (lk + 4 * q) * 17 + lr] = acc[y][q];
    __syncthreads();
    for (int e = threadIdx.x; e < 256; e += 64 * KW) {
      const int r = e >> 4, c = e & 15, j = t.j0 + 16 * y + c;
      double v = red[c * 17 + r];
#pragma unroll
      for (int w = 1; w < KW; w++) v += red[w * 272 + c * 17 + r];
      if (r < t.rn && j < nrhs) mv_apply<GM, T>(t, r, j, v, base[y], dpiv, W, V, Y, X, nrhs);
    }
  }
}

// Forward product task: 16 RT target rows, 16 NT right-hand sides, operand
// element (r, k) at a + r + k ld, the K range split over KW wave groups whose
// partial sums are added in group order, so a result never depends on
// scheduling.  Wave w takes the 16 target rows w mod RT and the K part w /
// RT.  Both operands go from memory straight into the registers of
// v_mfma_f64_16x16x4 (A operand: right-hand sides, B operand: target rows,
// 128 contiguous bytes per k), one CH-chunk ahead of their products; no
// staging and, for KW = 1, no barrier.  Loads are unconditional and in
// bounds: rows, columns and k past the task repeat its last one, their
// operand is set to zero or their result dropped.
// Bound by HBM: the operand is read once, and with 16 columns the matrix
// cores could take 19 TB/s.  KW = 4 reads 4.2-5.6 TB/s on fronts of 260 to
// 5544 pivot columns (a plain copy moves 5.05 here); 64-row tasks 2.1-5.0,
// 16 K parts 1.2-4.5 and only ahead when a level has few rows.
//
// GM = 1: the rows of W that a task adds to hold nothing yet; it takes what
// the front's (at most two) children add there, kids[row] being their rows of
// W (-1: none), instead of a launch before it.  GM = 2: it takes its source
// rows that way too, right-hand side row rsrc + k plus the children's, so that
// the level is one launch (GM_BYTES).
template <int NT, int RT, int KW, int GM, class T>
__global__ __launch_bounds__(64 * RT * KW) void k_fw(const MvTask* __restrict__ tasks, const T* __restrict__ pool,
                                                     const T* __restrict__ panel, const double* __restrict__ dpiv,
                                                     const int2* __restrict__ kids, double* W, double* V,
                                                     const double* R, double* Y, int nrhs) {
  static_assert(KW == 1 || RT == 1, "the K split works on 16-row tasks");
  constexpr int CH = NT == 1 && GM < 2 ? 32 : 16, ST = CH / 4;
  constexpr int NB = KW == 1 ? 4 * NT : NT;  // results of a thread
  const MvTask t = tasks[xcd_fours(blockIdx.x, gridDim.x)];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int r0 = 16 * (wv % RT), kw = wv / RT;
  if (KW == 1 && r0 >= t.rn) return;
  // this wave's K range, in whole chunks except at the end
  const int part = KW == 1 ? t.kn : (((t.kn + KW - 1) / KW + CH - 1) / CH) * CH;
  const int kb = kw * part, ke = min(t.kn, kb + part);
  const T* A = ((t.flags & MV_FRONT) ? pool : panel) + t.a + min(r0 + lr, t.rn - 1);
  int col[NT];
#pragma unroll
  for (int y = 0; y < NT; y++) col[y] = min(t.j0 + 16 * y + lr, nrhs - 1);
  const double* src = ((t.flags & MV_SRC_V) ? V : (t.flags & MV_SRC_R) ? R : W) + (int64_t)t.src * nrhs;
  f64x4 acc[NT];
#pragma unroll
  for (int y = 0; y < NT; y++) acc[y] = f64x4{0.0, 0.0, 0.0, 0.0};
  // row of W: the value at column c of the child's row q, 0.0 for none
  auto kid = [&](int q, int c) { return W[(int64_t)max(q, 0) * nrhs + c]; };
  // the children's part of this thread's results: rows first, values behind
  // the first operand loads
  double base[NB] = {}, add[2][NB];
  int2 own{-1, -1};
  const int erow = KW == 1 ? r0 + lr : (threadIdx.x >> 4) & 15;
  auto ecol = [&](int e) { return KW == 1 ? 16 * (e / 4) + lk + 4 * (e % 4) : 16 * e + ((int)threadIdx.x & 15); };
  if constexpr (GM > 0) own = kids[t.dst + min(erow, t.rn - 1)];
  auto load_base = [&]() {
    if constexpr (GM > 0)
#pragma unroll
      for (int e = 0; e < NB; e++) {
        const int c = min(t.j0 + ecol(e), nrhs - 1);
        add[0][e] = kid(own.x, c);
        add[1][e] = kid(own.y, c);
      }
  };
  struct Stage {
    T a[ST];
    double b[ST][NT], k0[GM == 2 ? ST : 1][NT], k1[GM == 2 ? ST : 1][NT];
    int2 q[GM == 2 ? ST : 1];
  };
  int2 next[GM == 2 ? ST : 1];  // the children's rows of the chunk that is loaded next
  auto load_kids = [&](int kc) {
    if constexpr (GM == 2)
#pragma unroll
      for (int s = 0; s < ST; s++) next[s] = kids[t.src + min(kc + 4 * s + lk, ke - 1)];
  };
  auto load = [&](int kc, Stage& g) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const int k = min(kc + 4 * s + lk, ke - 1);
      g.a[s] = A[(int64_t)k * t.ld];
      const double* b = GM == 2 ? R + (int64_t)(t.rsrc + k) * nrhs : src + (int64_t)k * nrhs;
#pragma unroll
      for (int y = 0; y < NT; y++) g.b[s][y] = b[col[y]];
    }
    if constexpr (GM == 2) {
#pragma unroll
      for (int s = 0; s < ST; s++) {
        g.q[s] = next[s];
#pragma unroll
        for (int y = 0; y < NT; y++) {
          g.k0[s][y] = kid(next[s].x, col[y]);
          g.k1[s][y] = kid(next[s].y, col[y]);
        }
      }
      load_kids(kc + CH);
    }
  };
  auto multiply = [&](int kc, const Stage& g) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const double a = kc + 4 * s + lk < ke ? (double)g.a[s] : 0.0;
#pragma unroll
      for (int y = 0; y < NT; y++) {
        double b = g.b[s][y];
        if constexpr (GM == 2) {
          b += g.q[s].x >= 0 ? g.k0[s][y] : 0.0;
          b += g.q[s].y >= 0 ? g.k1[s][y] : 0.0;
        }
        acc[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, acc[y], 0, 0, 0);
      }
    }
  };
  if (kb < ke) {
    Stage g0, g1;
    load_kids(kb);
    load(kb, g0);
    load_base();
    for (int kc = kb; kc < ke; kc += 2 * CH) {
      if (kc + CH < ke) load(kc + CH, g1);
      multiply(kc, g0);
      if (kc + CH >= ke) break;
      if (kc + 2 * CH < ke) load(kc + 2 * CH, g0);
      multiply(kc + CH, g1);
    }
  }
  if constexpr (GM > 0) {
    if (kb >= ke) load_base();
#pragma unroll
    for (int e = 0; e < NB; e++) base[e] = (own.x >= 0 ? add[0][e] : 0.0) + (own.y >= 0 ? add[1][e] : 0.0);
  }
  if constexpr (KW == 1) {
    // acc[y][q]: target row r0 + lr, right-hand side 16 y + lk + 4 q
    if (r0 + lr < t.rn)
#pragma unroll
      for (int y = 0; y < NT; y++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int j = t.j0 + 16 * y + lk + 4 * q;
          if (j < nrhs) mv_apply<GM, T>(t, r0 + lr, j, acc[y][q], base[4 * y + q], dpiv, W, V, Y, nullptr, nrhs);
        }
  } else {
    __shared__ double red[KW * 272];
    mv_combine<NT, KW, GM, T>(t, acc, base, red, dpiv, W, V, Y, nullptr, nrhs);
  }
}

// Backward product task: 16 target rows, operand element (r, k) at a + k +
// r ld (k contiguous), K split over KW waves as in k_fw.  A wave reads CH
// consecutive k of 64 / CH target rows a load and turns them through its own
// LDS tile into the MFMA operand, whose step s multiplies k = CH / 4 (lane /
// 16) + s.  GATHER: the source rows come through the fronts' row list (the
// first ky from Y, the others from X), else contiguous from W.  Operand and
// source rows are one chunk ahead of their products and the row list two, in
// that order, so that no load waits for a younger one.
template <bool GATHER, int NT, int KW, class T>
__global__ __launch_bounds__(64 * KW) void k_bw(const MvTask* __restrict__ tasks, const T* __restrict__ pool,
                                                const T* __restrict__ panel, const int* __restrict__ rows,
                                                double* W, double* Y, double* X, int nrhs) {
  constexpr int CH = NT <= 2 ? 32 : 16, ST = CH / 4, RPI = 64 / CH;
  // tile element (row, k) at row LT + 4 (k mod ST) + k / ST: conflict-free
  // reads by (lane mod 16, lane / 16)
  constexpr int LT = CH + 2, TILE = 16 * LT * (int)sizeof(T) / 8;
  __shared__ double lds[KW * (TILE > 272 ? TILE : 272)];
  const MvTask t = tasks[xcd_fours(blockIdx.x, gridDim.x)];
  const int lane = threadIdx.x & 63, kw = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  T* tile = reinterpret_cast<T*>(lds + kw * TILE);
  const int part = KW == 1 ? t.kn : (((t.kn + KW - 1) / KW + CH - 1) / CH) * CH;
  const int kb = kw * part, ke = min(t.kn, kb + part);
  const int ka = lane % CH, ia = lane / CH;  // this lane's k and first row of an operand load
  const T* A = ((t.flags & MV_FRONT) ? pool : panel) + t.a;
  int64_t arow[CH / 4];
#pragma unroll
  for (int q = 0; q < CH / 4; q++) arow[q] = (int64_t)min(q * RPI + ia, t.rn - 1) * t.ld;
  int col[NT];
#pragma unroll
  for (int y = 0; y < NT; y++) col[y] = min(t.j0 + 16 * y + lr, nrhs - 1);
  f64x4 acc[NT];
#pragma unroll
  for (int y = 0; y < NT; y++) acc[y] = f64x4{0.0, 0.0, 0.0, 0.0};
  T a[CH / 4];
  int idx[ST];
  double b[2][ST][NT];
  auto load_a = [&](int kc) {
    const T* p = A + min(kc + ka, ke - 1);
#pragma unroll
    for (int q = 0; q < CH / 4; q++) a[q] = p[arow[q]];
  };
  auto load_rows = [&](int kc) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const int k = min(kc + ST * lk + s, ke - 1);
      idx[s] = GATHER ? rows[t.src + k] : t.src + k;
    }
  };
  auto load_b = [&](int kc, double (&g)[ST][NT]) {
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const double* src = !GATHER ? W : min(kc + ST * lk + s, ke - 1) < t.ky ? Y : X;
      const double* r = src + (int64_t)idx[s] * nrhs;
#pragma unroll
      for (int y = 0; y < NT; y++) g[s][y] = r[col[y]];
    }
  };
  auto chunk = [&](int kc, double (&cur)[ST][NT], double (&nxt)[ST][NT]) {
    const bool in = kc + ka < ke;
#pragma unroll
    for (int q = 0; q < CH / 4; q++)
      tile[(q * RPI + ia) * LT + 4 * (ka % ST) + ka / ST] = in ? a[q] : (T)0;
    if (kc + CH < ke) {
      load_b(kc + CH, nxt);
      load_a(kc + CH);
      load_rows(min(kc + 2 * CH, ke - 1));
    }
    __builtin_amdgcn_wave_barrier();  // the tile is this wave's own: LDS keeps its order
#pragma unroll
    for (int s = 0; s < ST; s++) {
      const double av = (double)tile[lr * LT + 4 * s + lk];
#pragma unroll
      for (int y = 0; y < NT; y++) acc[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur[s][y], av, acc[y], 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  };
  if (kb < ke) {
    load_rows(kb);
    load_b(kb, b[0]);
    load_a(kb);
    load_rows(min(kb + CH, ke - 1));
    for (int kc = kb; kc < ke; kc += 2 * CH) {
      chunk(kc, b[0], b[1]);
      if (kc + CH < ke) chunk(kc + CH, b[1], b[0]);
    }
  }
  if constexpr (KW > 1) __syncthreads();  // the tiles' space takes the partial sums
  const double base[NT] = {};
  mv_combine<NT, KW, 0, T>(t, acc, base, lds, nullptr, W, nullptr, Y, X, nrhs);
}

// Forward-solve initialisation of the work rows of fronts with children, as
// far as the products do not gather them: row w takes the right-hand side row
// (pivot rows) plus the children's update rows that land in it, in child order.  Task: up to 64 work rows
// from w0, the first np of them pivot rows with right-hand side rows r0 ..
__global__ __launch_bounds__(1024) void k_fw_init(const InitTask* __restrict__ tasks, const int* __restrict__ gptr,
                                                  const int* __restrict__ gsrc, const double* __restrict__ R,
                                                  double* W, int nrhs) {
  const InitTask t = tasks[blockIdx.x];
  for (int idx = threadIdx.x; idx < t.rn * nrhs; idx += blockDim.x) {
    const int i = idx / nrhs, j = idx % nrhs, w = t.w0 + i;
    double v = i < t.np ? R[(int64_t)(t.r0 + i) * nrhs + j] : 0.0;
    const int e1 = gptr[w + 1];
    for (int e = gptr[w]; e < e1; e++) v += W[(int64_t)gsrc[e] * nrhs + j];
    W[(int64_t)w * nrhs + j] = v;
  }
}

template <int NT, class T>
static void mv_launch(hipStream_t st, const MvTask* t, int n, int kind, int kw, const T* pool, const T* panel,
                      const int* rows, const double* dpiv, const int2* kids, double* W, double* V, const double* R,
                      double* Y, double* X, int nrhs) {
  constexpr int KMAX = NT == 1 ? 16 : 8;  // registers: a 1024-thread workgroup has 128 a lane
  auto bw = [&](auto g) {
    constexpr bool G = decltype(g)::value;
    if (kw == 1) k_bw<G, NT, 1, T><<<n, 64, 0, st>>>(t, pool, panel, rows, W, Y, X, nrhs);
    else if (kw == 4) k_bw<G, NT, 4, T><<<n, 256, 0, st>>>(t, pool, panel, rows, W, Y, X, nrhs);
    else k_bw<G, NT, KMAX, T><<<n, 64 * KMAX, 0, st>>>(t, pool, panel, rows, W, Y, X, nrhs);
  };
  auto fw = [&](auto g) {
    constexpr int GM = decltype(g)::value;
    if (kw == 1) k_fw<NT, 4, 1, GM, T><<<n, 256, 0, st>>>(t, pool, panel, dpiv, kids, W, V, R, Y, nrhs);
    else if (kw == 4) k_fw<NT, 1, 4, GM, T><<<n, 256, 0, st>>>(t, pool, panel, dpiv, kids, W, V, R, Y, nrhs);
    else k_fw<NT, 1, KMAX, GM, T><<<n, 64 * KMAX, 0, st>>>(t, pool, panel, dpiv, kids, W, V, R, Y, nrhs);
  };
  if (kind == MV_FORWARD) {
    fw(std::integral_constant<int, 0>{});
  } else if (kind == MV_FORWARD_ADD) {
    fw(std::integral_constant<int, 1>{});
  } else if (kind == MV_FORWARD_ALL) {
    if constexpr (NT <= GM_TILES) fw(std::integral_constant<int, 2>{});
  } else if (kind == MV_BACK_ROWS) {
    bw(std::true_type{});
  } else {
    bw(std::false_type{});
  }
}

#define FGPU_MV(T)                                                                                                 \
  void launch_mv(hipStream_t st, const MvTask* t, int n, int kind, int nt, int kw, const T* pool, const T* panel,  \
                 const int* rows, const double* dpiv, const int2* kids, double* W, double* V, const double* R,     \
                 double* Y, double* X, int nrhs) {                                                                 \
    if (n <= 0) return;                                                                                            \
    switch (nt) {                                                                                                  \
      case 1: mv_launch<1, T>(st, t, n, kind, kw, pool, panel, rows, dpiv, kids, W, V, R, Y, X, nrhs); break;      \
      case 2: mv_launch<2, T>(st, t, n, kind, kw, pool, panel, rows, dpiv, kids, W, V, R, Y, X, nrhs); break;      \
      case 3: mv_launch<3, T>(st, t, n, kind, kw, pool, panel, rows, dpiv, kids, W, V, R, Y, X, nrhs); break;      \
      case 4: mv_launch<4, T>(st, t, n, kind, kw, pool, panel, rows, dpiv, kids, W, V, R, Y, X, nrhs); break;      \
      case 5: mv_launch<5, T>(st, t, n, kind, kw, pool, panel, rows, dpiv, kids, W, V, R, Y, X, nrhs); break;      \
      default: mv_launch<6, T>(st, t, n, kind, kw, pool, panel, rows, dpiv, kids, W, V, R, Y, X, nrhs); break;     \
    }                                                                                                              \
  }
FGPU_MV(double)
FGPU_MV(float)
#undef FGPU_MV

void launch_fw_init(hipStream_t st, const InitTask* t, int n, const int* gptr, const int* gsrc, const double* R,
                    double* W, int nrhs) {
  if (n > 0) k_fw_init<<<n, std::min(1024, ((64 * nrhs + 63) / 64) * 64), 0, st>>>(t, gptr, gsrc, R, W, nrhs);
}

}  // namespace fgpu
