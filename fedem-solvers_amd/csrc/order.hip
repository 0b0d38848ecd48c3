// Change of order between the callers' vectors (column-major, equations in
// SAM order) and the reducer's (row-major, rows in elimination order), on the
// device, so that a vector crosses the bus once and the host does not touch
// it; and the gathered upload of arrays.
#include "kern_device.hpp"

namespace fgpu {

// A workgroup takes 64 source rows by 16 columns through an LDS tile: the
// column-major side in runs of 64 rows, the row-major side in runs of 16
// columns.  Bound by HBM, far below the copy over the bus.  With the order on
// the host a solve of 40,404 equations by 33 columns took 3.6 ms, now 1.5, and
// 7 load cases with their recovery on 38,000 equations 1.9, now 0.67.
constexpr int OT_ROWS = 64, OT_COLS = 16;

// out[map[q]][c] = in[q + c ldi] (map null: row q itself)
__global__ __launch_bounds__(256) void k_rows_in(int n, int nc, const int* __restrict__ map,
                                                 const double* __restrict__ in, int64_t ldi, double* __restrict__ out,
                                                 int ldo) {
  __shared__ double tile[OT_COLS][OT_ROWS + 1];
  const int q0 = blockIdx.x * OT_ROWS, c0 = blockIdx.y * OT_COLS;
  const int rows = min(OT_ROWS, n - q0), cols = min(OT_COLS, nc - c0);
  for (int e = threadIdx.x; e < OT_ROWS * cols; e += 256) {
    const int q = e & (OT_ROWS - 1), c = e / OT_ROWS;
    if (q < rows) tile[c][q] = in[q0 + q + (int64_t)(c0 + c) * ldi];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < OT_ROWS * OT_COLS; e += 256) {
    const int c = e % OT_COLS, q = e / OT_COLS;
    if (q < rows && c < cols) out[(int64_t)(map ? map[q0 + q] : q0 + q) * ldo + c0 + c] = tile[c][q];
  }
}

// out[q + c ldo] = A[map[q]][c] + B[map[q]][c], either of which may be null
__global__ __launch_bounds__(256) void k_rows_out(int n, int nc, const int* __restrict__ map,
                                                  const double* __restrict__ A, int lda, const double* __restrict__ B,
                                                  int ldb, double* __restrict__ out, int64_t ldo) {
  __shared__ double tile[OT_COLS][OT_ROWS + 1];
  const int q0 = blockIdx.x * OT_ROWS, c0 = blockIdx.y * OT_COLS;
  const int rows = min(OT_ROWS, n - q0), cols = min(OT_COLS, nc - c0);
  for (int e = threadIdx.x; e < OT_ROWS * OT_COLS; e += 256) {
    const int c = e % OT_COLS, q = e / OT_COLS;
    if (q < rows && c < cols) {
      const int64_t r = map[q0 + q];
      double v = A ? A[r * lda + c0 + c] : 0.0;
      if (B) v = A ? v + B[r * ldb + c0 + c] : B[r * ldb + c0 + c];
      tile[c][q] = v;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < OT_ROWS * cols; e += 256) {
    const int q = e & (OT_ROWS - 1), c = e / OT_ROWS;
    if (q < rows) out[q0 + q + (int64_t)(c0 + c) * ldo] = tile[c][q];
  }
}

// The column tiles of a launch go in grid rows of at most 65,535.
template <class F>
static void by_columns(int n, int nc, F&& go) {
  constexpr int most = 65535 * OT_COLS;
  if (n > 0)
    for (int c0 = 0; c0 < nc; c0 += most) {
      const int k = nc - c0 < most ? nc - c0 : most;
      go(dim3(nblk(n, OT_ROWS), nblk(k, OT_COLS)), c0, k);
    }
}

void launch_rows_in(hipStream_t st, int n, int nc, const int* map, const double* in, int64_t ldi, double* out,
                    int ldo) {
  by_columns(n, nc, [&](dim3 g, int c0, int k) {
    k_rows_in<<<g, 256, 0, st>>>(n, k, map, in + c0 * ldi, ldi, out + c0, ldo);
  });
}

void launch_rows_out(hipStream_t st, int n, int nc, const int* map, const double* A, int lda, const double* B, int ldb,
                     double* out, int64_t ldo) {
  by_columns(n, nc, [&](dim3 g, int c0, int k) {
    k_rows_out<<<g, 256, 0, st>>>(n, k, map, A ? A + c0 : nullptr, lda, B ? B + c0 : nullptr, ldb, out + c0 * ldo, ldo);
  });
}

// (Here and not beside the scratch array of the load vectors without
// allocation, whose code object a program would load with its first load case:
// 13 ms and 32 MiB.)
// Fred (nd x nrhs, column-major) = [r2 rows in dofPosIn2 order; r1; 0]
__global__ void k_scatter_reduced(int nd, int n2, int ngen, int nrhs, const int* __restrict__ pos2,
                                  const double* __restrict__ r2, const double* __restrict__ r1,
                                  double* __restrict__ Fred) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)nd * nrhs) return;
  const int i = (int)(g % nd), c = (int)(g / nd);
  double v = 0.0;
  if (i < n2) v = r2[(int64_t)(pos2[i] - 1) * nrhs + c];
  else if (i < n2 + ngen) v = r1[(int64_t)(i - n2) * nrhs + c];
  Fred[g] = v;
}

void launch_scatter_reduced(hipStream_t st, int nd, int n2, int ngen, int nrhs, const int* pos2, const double* r2,
                            const double* r1, double* Fred) {
  const int64_t n = (int64_t)nd * nrhs;
  if (n > 0) k_scatter_reduced<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(nd, n2, ngen, nrhs, pos2, r2, r1, Fred);
}

// One workgroup per block of a gathered upload, table and data read straight
// from pinned host memory: 16 bytes a load, two in flight per thread, the last
// words of an array one by one (blocks start at multiples of 16 on both sides).
__global__ __launch_bounds__(256) void k_copy_blocks(const CopyBlock* __restrict__ table, const char* __restrict__ stage) {
  const CopyBlock b = table[blockIdx.x];
  const uint4* in = reinterpret_cast<const uint4*>(stage + b.from);
  uint4* out = static_cast<uint4*>(b.dst);
  const unsigned n = b.bytes / 16;
#pragma unroll 2
  for (unsigned i = threadIdx.x; i < n; i += 256) out[i] = in[i];
  const unsigned w = 4 * n + threadIdx.x;
  if (w < b.bytes / 4) reinterpret_cast<unsigned*>(out)[w] = reinterpret_cast<const unsigned*>(in)[w];
}

void launch_copy_blocks(hipStream_t st, int n, const CopyBlock* table, const char* stage) {
  if (n > 0) k_copy_blocks<<<n, 256, 0, st>>>(table, stage);
}

}  // namespace fgpu
