// Shared device-side declarations for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace fgpu {

// Dense multi-vectors (right-hand sides, B columns, Lanczos blocks) are stored
// row-major: V[row * nrhs + j], so that one matrix row is contiguous.
//
// A factorisation task list entry.  The host builds one list per level and
// panel step; see reducer_gpu.cpp.
struct FTask {
  int sn;      // supernode
  int a, b;    // meaning depends on the kernel (row chunk, tile indices)
  int k0;      // first pivot column of the panel
  int kb;      // trailing update: panel width (<= 256); the trailing block starts at k0 + kb
  int je;      // trailing update: columns from je on are left alone (0: none)
};

// Elements that the solve-panel pools hold past their last front: k_panel's
// 16-byte loads may run on past a column.
constexpr int PANEL_PAD = 4;

// A solve product task (solve.hip): target rows x right-hand sides j0 .. from
// the operand at a (leading dimension ld) and kn source rows.
struct MvTask {
  int64_t a;   // offset of the operand's first element in the solve panels or (MV_FRONT) the fronts
  int ld;
  int rn, kn;  // target rows (<= 64) and source rows
  int src;     // first source row, or (MV_BACK_ROWS) first entry of the fronts' row list
  int ky;      // MV_BACK_ROWS: the first ky source rows are rows of Y, the others of X
  int dst;     // first target row
  int dst2;    // MV_Y: first row of V to keep the result in (-1: none); MV_YSUB: first row of Y
  int flags;
  int j0;
  int rsrc;    // MV_FORWARD_ALL: first right-hand side row of the source rows
};
// A level whose products read up to GM_BYTES of source rows gathers them itself
// (up to three times the reads against a launch less), with up to GM_TILES
// 16-column groups (registers).  Limits of 32 and 200 MiB came out the same to
// 0.5 % from the 17x13x11 to the 45x41x43 block; the one that reads least stands.
constexpr int64_t GM_BYTES = 8 << 20;
constexpr int GM_TILES = 2;
enum MvKind : int {
  MV_FORWARD,      // operand rows contiguous
  MV_FORWARD_ADD,  // the same, MV_ADD and MV_SUB targets gathered from the children
  MV_FORWARD_ALL,  // source rows gathered from right-hand sides and children as well (up to GM_TILES column groups)
  MV_BACK_ROWS,    // operand k contiguous, source rows through the fronts' row list
  MV_BACK          // operand k contiguous, source rows contiguous in W
};
enum MvFlags : int {
  MV_FRONT = 1,                  // operand in the fronts (L21), not the solve panels
  MV_SRC_V = 2, MV_SRC_R = 4,    // source rows in V or R, not W
  MV_APPLY = 0xf0,
  MV_Y = 0x10,                   // Y = v / D (and V = v)
  MV_SET = 0x20, MV_NEG = 0x30,  // W = v, W = -v
  MV_ADD = 0x40, MV_SUB = 0x50,  // W += v, W -= v
  MV_X = 0x60,                   // X = v
  MV_YSUB = 0x70                 // W = Y - v (Y may be absent: zero)
};

// Forward initialisation of up to 64 work rows from w0 (k_fw_init).
struct InitTask {
  int w0, rn;
  int np, r0;  // the first np rows are pivot rows, with right-hand side rows r0 ..
};

struct DevSym {
  const int* col0;
  const int* ncol;
  const int* nrow;
  const int64_t* foff;
  const int* rptr;
  const int* rows;
  const int* chptr;
  const int* chlist;
  const int* relptr;
  const int* rel;
  const int* ild;       // per-front leading dimension of the solve panel (nrow in fused levels, else ncol)
  double* dpiv;         // pivots D of the LDL^T factor by pivot column (col0[front] + column)
  // singular pivots: a pivot d_j with |d_j| <= tolf |a_jj| (a_jj the
  // original diagonal, adiag) is replaced by |a_jj| (by amax when a_jj = 0)
  // and its column flagged in sing: 1 a true zero (|d_j| at rounding level
  // of a_jj, or a_jj = 0), 2 a pivot reduced to near zero
  const double* adiag;
  const double* amax;
  int* sing;
  double tolf;
};

}  // namespace fgpu
