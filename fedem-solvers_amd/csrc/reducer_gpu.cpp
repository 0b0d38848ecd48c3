// Device orchestration of one part reduction on a single MI355X.
//
// Phase map to the reference driver (reducer.f90:22-748):
//   elements + assembly   INADD / csAddEM                    (inadd.f90:26-464)
//   factor + Schur        csSolveSupEl SPR branch, SPRFC1 +
//                         SPREXK                              (solExtensionModule.f90:708-775)
//   B                     SPRBS1/2 per external DOF           (solExtensionModule.f90:809-843)
//   component modes       EIGVAL -> csLanczosEigenSolve       (cmstrs.f90:53-263)
//   mass / stiffness      CMSTRS K11, M11, M12, M22           (cmstrs.f90:728-944)
//   gravity               GRAVfull + GRAV                     (cmstrs.f90:286-474)
//   dispfile              vgi = K_ii^{-1} g_i                 (cmstrs.f90:674-712)
#include "reducer_gpu.hpp"
#include <algorithm>
#include <atomic>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <future>
#include <mutex>
#include "dense_small.hpp"
#include "host_jobs.hpp"
#include "kernels.hpp"

namespace fgpu {

#define HIPCHK(x)                                                                          \
  do {                                                                                     \
    hipError_t e_ = (x);                                                                   \
    if (e_ != hipSuccess) {                                                                \
      err = std::string("HIP error '") + hipGetErrorString(e_) + "' in " + #x;             \
      return -3;                                                                           \
    }                                                                                      \
  } while (0)

// Device bytes held by the buffers that the calling thread allocates (the
// server gives every slot's worker thread its own counter).
static thread_local std::atomic<int64_t>* tl_account = nullptr;
void set_alloc_account(std::atomic<int64_t>* a) { tl_account = a; }
// Stream the uploads of this thread go through (the handle's own stream while
// one of its methods runs), so that they never wait for other handles' work
// the way copies on the null stream would.
static thread_local hipStream_t tl_stream = nullptr;
struct StreamScope {
  hipStream_t prev;
  explicit StreamScope(hipStream_t s) : prev(tl_stream) { tl_stream = s; }
  ~StreamScope() { tl_stream = prev; }
};

// Pinned host memory that no handle of the process uses, for the next one that
// asks for as much on the same device: a call for it takes 11-15 us, every so
// often 60-330 (a new mapping, whose pages are then touched for the first
// time), and as much to give it back.  Blocks are powers of two; at most MOST
// bytes stay here, the others go back to the system.  One object for the
// process, never destroyed (at its end the runtime may be gone before it).
class PinnedPool {
 public:
  static PinnedPool& get() {
    static PinnedPool* pool = new PinnedPool;
    return *pool;
  }
  hipError_t take(size_t bytes, void** p, int* dev) {
    if (hipError_t e = hipGetDevice(dev)) return e;
    {
      std::lock_guard<std::mutex> g(mu_);
      for (size_t k = 0; k < idle_.size(); k++)
        if (idle_[k].bytes == bytes && idle_[k].dev == *dev) {
          *p = idle_[k].p;
          held_ -= bytes;
          idle_.erase(idle_.begin() + k);
          return hipSuccess;
        }
    }
    return hipHostMalloc(p, bytes, hipHostMallocDefault);
  }
  // no work of the device on the block may be outstanding
  void give(void* p, size_t bytes, int dev) {
    {
      std::lock_guard<std::mutex> g(mu_);
      if (held_ + bytes <= MOST) {
        try {
          idle_.push_back({p, bytes, dev});
          held_ += bytes;
          return;
        } catch (const std::bad_alloc&) {
        }
      }
    }
    (void)hipHostFree(p);
  }

 private:
  static constexpr size_t MOST = 8 << 20;
  struct Block {
    void* p;
    size_t bytes;
    int dev;
  };
  std::mutex mu_;
  std::vector<Block> idle_;
  size_t held_ = 0;
};

// Pinned host memory for asynchronous copies.  Growing it waits for the
// thread's stream; an owner that releases it has waited for its own.
template <class T>
struct HBuf {
  T* p = nullptr;
  size_t n = 0;
  HBuf() = default;
  HBuf(const HBuf&) = delete;
  HBuf& operator=(const HBuf&) = delete;
  ~HBuf() { release(); }
  void release() {
    if (p) PinnedPool::get().give(p, bytes_, dev_);
    p = nullptr;
    n = 0;
  }
  hipError_t alloc(size_t count) {
    if (count <= n && p) return hipSuccess;
    if (p && tl_stream)
      if (hipError_t e = hipStreamSynchronize(tl_stream)) return e;
    release();
    bytes_ = 4096;
    while (bytes_ < count * sizeof(T)) bytes_ *= 2;
    const hipError_t e = PinnedPool::get().take(bytes_, (void**)&p, &dev_);
    if (e == hipSuccess) n = count;
    else p = nullptr;
    return e;
  }

 private:
  size_t bytes_ = 0;
  int dev_ = 0;
};

// Two pieces of pinned memory through which arrays go to and from the device:
// the host fills or reads one while the device reads or fills the other.
struct Stage {
  static constexpr size_t PIECE = 512 << 10;
  HBuf<char> mem;
  hipEvent_t event[2]{};
  enum { FREE, EVENT, STREAM } until[2]{};  // what the device's work on a piece ends with
  hipStream_t stream = nullptr;

  ~Stage() {
    for (hipEvent_t& e : event)
      if (e) (void)hipEventDestroy(e);
  }
  hipError_t open() {
    if (mem.p) return hipSuccess;
    for (hipEvent_t& ev : event)
      if (!ev)
        if (hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) return e;
    return mem.alloc(2 * PIECE);
  }
  char* piece(int h) { return mem.p + h * PIECE; }
  // The device's work on piece h is what the stream has been given so far.
  // Without an event of its own (which costs the stream some 5 us) where the
  // stream is waited for anyway before the piece is wanted again.
  hipError_t mark(int h, hipStream_t st, bool own_event = true) {
    stream = st;
    until[h] = own_event ? EVENT : STREAM;
    return own_event ? hipEventRecord(event[h], st) : hipSuccess;
  }
  // piece h is the host's again
  hipError_t wait(int h) {
    const auto u = until[h];
    until[h] = FREE;
    if (u == STREAM) return hipStreamSynchronize(stream);
    return u == EVENT ? hipEventSynchronize(event[h]) : hipSuccess;
  }
  // the stream has been waited for
  void passed() { until[0] = until[1] = FREE; }
};

// Arrays on their way to the device.  While a batch is open on the thread its
// uploads are gathered in the stage's pieces, behind a table of blocks of up to
// 8 KB; a kernel reads a full piece and writes its blocks while the host fills
// the other, flush() sends what is there.  Each array is uploaded once and
// kept until the batch ends.  An array by itself costs a staged copy and a
// wait, 15 us each (0.8 of the 1.46 ms in which a 20x10 plate was analysed,
// uploaded and reduced; 0.69 in all with its 45 small arrays gathered), and a
// large one goes through staging memory of the runtime's own, whose pages are
// new with most handles: 2.4 GB/s, until 16 MB have passed.
struct UploadBatch {
  static constexpr size_t TABLE = 16 << 10, MOST = TABLE / sizeof(CopyBlock), DATA = Stage::PIECE - TABLE;
  Stage& stage;
  hipStream_t st = nullptr;
  hipError_t err = hipSuccess;
  int h = 0;
  size_t used = 0, blocks = 0;

  explicit UploadBatch(Stage& s) : stage(s) {}
  hipError_t open(hipStream_t s) {
    st = s;
    err = stage.open();
    used = blocks = 0;
    return err;
  }
  hipError_t put(void* dst, const void* src, size_t bytes) {
    for (size_t o = 0; o < bytes && err == hipSuccess;) {
      const size_t n = std::min({bytes - o, DATA - used, (MOST - blocks) * COPY_BLOCK});
      if (n == 0) {
        (void)flush(true);  // (err)
        continue;
      }
      if (blocks == 0 && (err = stage.wait(h)) != hipSuccess) break;
      CopyBlock* t = reinterpret_cast<CopyBlock*>(stage.piece(h));
      std::memcpy(stage.piece(h) + TABLE + used, static_cast<const char*>(src) + o, n);
      for (size_t q = 0; q < n; q += COPY_BLOCK)
        t[blocks++] = {static_cast<char*>(dst) + o + q, (unsigned)(TABLE + used + q),
                       (unsigned)std::min(COPY_BLOCK, n - q)};
      used = std::min(DATA, (used + n + 15) & ~(size_t)15);
      o += n;
    }
    return err;
  }
  hipError_t flush(bool full = false) {
    if (blocks == 0 || err != hipSuccess) return err;
    launch_copy_blocks(st, (int)blocks, reinterpret_cast<const CopyBlock*>(stage.piece(h)), stage.piece(h));
    used = blocks = 0;
    err = hipGetLastError();
    if (err == hipSuccess) err = stage.mark(h, st, full);
    h ^= 1;
    return err;
  }
};
static thread_local UploadBatch* tl_batch = nullptr;
struct BatchScope {
  explicit BatchScope(UploadBatch& b) { tl_batch = &b; }
  ~BatchScope() {
    (void)tl_batch->flush();
    tl_batch = nullptr;
  }
};

template <class T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  std::atomic<int64_t>* acct = nullptr;  // counter charged with this buffer
  DBuf() = default;
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  ~DBuf() { release(); }
  void release() {
    if (p) {
      (void)hipFree(p);
      if (acct) *acct -= (int64_t)(std::max<size_t>(1, n) * sizeof(T));
    }
    p = nullptr;
    n = 0;
    acct = nullptr;
  }
  hipError_t alloc(size_t count) {
    if (count <= n && p) return hipSuccess;
    release();
    hipError_t e = hipMalloc((void**)&p, std::max<size_t>(1, count) * sizeof(T));
    if (e != hipSuccess) {
      p = nullptr;
      return e;
    }
    n = count;
    acct = tl_account;
    if (acct) *acct += (int64_t)(std::max<size_t>(1, n) * sizeof(T));
    return hipSuccess;
  }
  hipError_t upload(const std::vector<T>& v) {
    hipError_t e = alloc(v.size());
    if (e != hipSuccess || v.empty()) return e;
    static_assert(sizeof(T) % 4 == 0, "a batch moves whole words");
    if (tl_batch) return tl_batch->put(p, v.data(), v.size() * sizeof(T));
    if (!tl_stream) return hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
    e = hipMemcpyAsync(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, tl_stream);
    return e == hipSuccess ? hipStreamSynchronize(tl_stream) : e;  // v may go out of scope after the call
  }
};

enum OpKind {
  FRONT_ZERO,  // the first of the factor schedule, issued before the assembly
  EXTADD, DIAG, TRSM, DIAG_TRSM, UPDATE, INV_MUL, PANEL,
  UPDATE_SIDE, FORK, JOIN,  // lookahead: trailing tiles on the side stream, fork/join with the main one
  FW_INIT, FW_MV, FW_MV_ADD, FW_MV_ALL, BW_ROWS, BW_MV  // solve plans
};
struct Op {
  int kind, off, n;
  int kw = 1;  // solve products: K parts per workgroup; extend-add: rows of the largest front
};

// Where the solve panels lie and which levels are fused (solve.hip).
struct SolveLayout {
  std::vector<char> fused;    // per level
  std::vector<int64_t> ioff;  // per front (nsup + 1)
  std::vector<int> ild;       // per front
  bool unfused = false;       // some level with fronts is not fused (its solves need V)
};

struct SolvePlan {
  bool valid = false;  // built for the current structure
  int nrhs = 0, nt = 1;  // 16-column groups of right-hand sides per task
  std::vector<Op> fw, bw, bw0;  // bw0: from a zero Y (displacement recovery matrix B)
  DBuf<MvTask> tasks;
  DBuf<InitTask> inits;
};

// Host lists of a solve plan before their upload.
struct PlanHost {
  std::vector<MvTask> tasks;
  std::vector<InitTask> inits;
};

// A captured launch sequence (HIP graph), replayed while the buffers it
// was captured with are unchanged (key = their addresses).
struct GraphCache {
  hipGraphExec_t exec = nullptr;
  std::vector<const void*> key;
  void reset() {
    if (exec) (void)hipGraphExecDestroy(exec);
    exec = nullptr;
    key.clear();
  }
  ~GraphCache() { reset(); }
};

// Replays gc when its key matches, else captures body() on stream st (kernel
// launches only: no memset or host-synchronous call inside) and launches it.
template <class F>
static hipError_t run_graph(hipStream_t st, GraphCache& gc, const std::vector<const void*>& key, F&& body) {
  if (gc.exec && gc.key == key) return hipGraphLaunch(gc.exec, st);
  if (gc.exec) {
    (void)hipGraphExecDestroy(gc.exec);
    gc.exec = nullptr;
  }
  hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) return e;
  body();
  hipGraph_t g = nullptr;
  e = hipStreamEndCapture(st, &g);
  if (e != hipSuccess) return e;
  e = hipGraphInstantiate(&gc.exec, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e != hipSuccess) {
    gc.exec = nullptr;
    return e;
  }
  gc.key = key;
  return hipGraphLaunch(gc.exec, st);
}

struct DeviceReducer::Impl {
  GraphCache g_factor;
  Stage stage;
  UploadBatch batch{stage};
  DBuf<int> sb_cnt, sb_tsum, sb_bad;  // the structure build's counts
  int factor_runs = 0;  // factorisations since the last upload
  // part
  DBuf<double> xyz, eprop;
  DBuf<int> eptr, enodes, hexlist, shlist, bmlist, p1;
  DBuf<int64_t> eoff;
  // structure
  DBuf<int> col0, ncol, nrow, rptr, rows, chptr, chlist, relptr, rel, rowptr, colind, cptr, cidx;
  DBuf<int64_t> foff, fmap, ioff;
  DBuf<int> ild;
  SolveLayout lay;
  DBuf<int> gptr, gsrc;  // forward init: the child update rows added to each work row, in child order
  DBuf<int2> kids;       // the first two of them (-1: none)
  // inputs of the device structure build: SAM arrays, element types, per
  // node first equation / equation count / neighbour lists (+ DOF offsets),
  // per row its node, per column its front
  DBuf<int> madof, msc, nndof, drank, etype, nfirst, neqd, nbptr, nbl, nbo, rnode, colsn;
  DBuf<double> signs;                    // mode signs and the per-group bests of their search
  // grow-only work arrays of the load-case calls (freeing device memory
  // waits for the whole device, so they are kept between calls)
  DBuf<double> sk_r, sk_t, sk_x, rl_f, rc_s, rc_y, gi_g;
  DBuf<int> ceq_ptr, ceq_node, ceq_dof;  // constraint equations of the dependent DOFs
  DBuf<double> ceq_coef;
  DBuf<int> e2p, pos2;  // perm row of every equation; dofPosIn2 (for the device-side reduced loads)
  DevSym S{};
  DBuf<FTask> ftasks;
  DBuf<int> xrange;  // extend-add tasks: (child, first, end) column ranges
  DBuf<double> dpiv;   // pivots D of the factor by pivot column (FP64 for both factor types)
  DBuf<double> adiag, amax;  // original (mixed: equilibrated) diagonal of K_ii and its largest magnitude
  DBuf<int> sing;            // per pivot column: 0, 1 true zero replaced, 2 reduced-to-zero replaced
  DBuf<double> itmp;  // products of the pairs that the pivot-block inverses are joined from (FP32 ones use half)
  std::vector<Op> fops;
  std::map<int, std::unique_ptr<SolvePlan>> plans;
  // values
  DBuf<double> Kp, Mp, Kv, Mv, pool, W, V, ipool;
  DBuf<int> ebad, piv;
  DBuf<double> X, Z, Y, part, small, acc, grav, ccoef;
  DBuf<double> emass;  // nel element masses, then their total
  // mixed precision: FP32 fronts and pivot-block inverses, equilibration
  // scale, refinement residual and norm partials
  bool mixed = false;
  bool m_diag = false;  // only lumped-mass (ANDES4) elements and no constraints: M is diagonal in a K-shaped pattern
  DBuf<int> row0, dpos;  // first row of every node (in row order), place of every row's diagonal
  int nnode = 0;
  NodeRows node_rows(int nrow) const { return {row0.p, nnode, nrow}; }
  int solve_split = 128;
  DBuf<float> pool32, ipool32;
  DBuf<double> dscale, dcs, Rr, irpart;
  DBuf<double> cg_p, cg_q, cg_z, cg_t, cg_part, cg_dot, cg_co;  // conjugate-gradient refinement
  std::vector<double> s22;  // mixed: Schur complement from the refined B (n2 x n2, column-major)
  // component modes
  DBuf<double> Q, P, Wl, Zl, Yl, Cc, Phi, Tmp;
  // a Lanczos step's record for the host: the breakdown flag (an int in the
  // first entry), the two CholQR factors, the reorthogonalisation
  // coefficients; two pinned copies (step parity)
  DBuf<double> lzrec;
  HBuf<double> hrec;
  HBuf<int> hpiv;     // the pivot statistics and
  HBuf<double> hred;  // the reduced matrices on their way to the host
  hipEvent_t lz_ev[2]{};
  hipStream_t side = nullptr;  // lookahead stream of the factorisation
  hipEvent_t fj[2]{};          // its fork and join events
  std::vector<int> hexl, shl, bml;  // elements by type: HEX8, ANDES4, BEAM2
  int64_t wrows = 0;
  hipEvent_t ev[12]{};
  std::vector<hipEvent_t> upd_ev;  // start/stop pairs of the trailing-update launches
};

DeviceReducer::DeviceReducer() : d_(new Impl) {}
DeviceReducer::~DeviceReducer() {
  if (st_) {
    (void)hipStreamSynchronize(st_);
    for (auto& e : d_->ev)
      if (e) (void)hipEventDestroy(e);
    for (auto& e : d_->upd_ev) (void)hipEventDestroy(e);
    for (auto& e : d_->lz_ev)
      if (e) (void)hipEventDestroy(e);
    for (auto& e : d_->fj)
      if (e) (void)hipEventDestroy(e);
    if (d_->side) {
      (void)hipStreamSynchronize(d_->side);
      (void)hipStreamDestroy(d_->side);
    }
    (void)hipStreamDestroy(st_);
  }
}

// Solve panels of the fronts.  A level is fused (its Y21 = -L21 L11^-1
// formed, one product per pass instead of two) when forming Y21 costs less
// than the launches saved: sum nu nc^2 flops at about 40 TFLOP/s against
// some 12 us for each pass pair, over the solves that the handle's options
// let expect (block Lanczos 16, mixed-precision refinement 8, else B and one
// load-case solve).
static SolveLayout solve_layout(const Symbolic& y, const ReduceOptions& o) {
  SolveLayout q;
  const double nsolve = o.ngen > 0 ? 16 : o.mixed ? 8 : 2;
  q.fused.assign(y.nlevels, 1);
  q.ild.assign(y.nsup, 0);
  q.ioff.assign(y.nsup + 1, 0);
  for (int l = 0; l < y.nlevels; l++) {
    double flops = 0.0;
    bool any = false;
    for (int k = y.lvptr[l]; k < y.lvptr[l + 1]; k++) {
      const int s = y.lvsup[k];
      const double nc = y.ncol[s], nu = y.nrow[s] - nc;
      flops += nu * nc * nc;
      any = any || nc > 0;
    }
    q.fused[l] = flops <= nsolve * 4.8e8;
    if (any && !q.fused[l]) q.unfused = true;
    for (int k = y.lvptr[l]; k < y.lvptr[l + 1]; k++) {
      const int s = y.lvsup[k];
      q.ild[s] = q.fused[l] ? y.nrow[s] : y.ncol[s];
    }
  }
  for (int s = 0; s < y.nsup; s++) q.ioff[s + 1] = q.ioff[s] + (int64_t)q.ild[s] * y.ncol[s];
  return q;
}

// Elements of the products that the pivot-block inverses of all fronts are
// joined from, pairs of h tiles at a time (k_inv_mul): the most of any h, in
// units of the 16 elements that a task counts by.
static int64_t inverse_products(const Symbolic& y, int h, int s) {
  int64_t units = 0;
  for (int m = h; 64 * m < y.ncol[s]; m += 2 * h) units += 4 * h * (std::min(64 * (m + h), y.ncol[s]) - 64 * m);
  return units;
}
static int64_t inverse_workspace(const Symbolic& y) {
  int64_t most = 0;
  int maxc = 0;
  for (int s = 0; s < y.nsup; s++) maxc = std::max(maxc, y.ncol[s]);
  for (int h = 1; 64 * h < maxc; h *= 2) {
    int64_t all = 0;
    for (int s = 0; s < y.nsup; s++) all += inverse_products(y, h, s);
    most = std::max(most, 16 * all);
  }
  return most;
}

static void build_factor_schedule(const Symbolic& y, const SolveLayout& lay, std::vector<FTask>& tasks,
                                  std::vector<Op>& ops, std::vector<int>& xrange, double& flops, int panel,
                                  bool lookahead) {
  xrange.clear();
  std::vector<int> at;
  flops = 0;
  // columns of a front cleared before the original entries go in (k_front_zero),
  // the largest fronts first
  auto own = [&](int s) { return y.chptr[s + 1] == y.chptr[s] || s == y.nsup - 1 ? y.nrow[s] : y.ncol[s]; };
  for (int s = y.nsup - 1; s >= 0; s--)
    for (int j0 = 0; j0 < own(s); j0 += 16) tasks.push_back({s, j0, 0, own(s), 0, 0});
  ops.push_back({FRONT_ZERO, 0, (int)tasks.size()});
  for (int l = 0; l < y.nlevels; l++) {
    const int* sups = &y.lvsup[y.lvptr[l]];
    const int ns = y.lvptr[l + 1] - y.lvptr[l];
    int off = (int)tasks.size(), rows = 0;
    for (int q = 0; q < ns; q++) {
      int s = sups[q];
      if (y.chptr[s + 1] == y.chptr[s]) continue;
      rows = std::max(rows, y.nrow[s]);
      // extend-add task (front s, 16-column block j0): the (child, first,
      // end) ranges of child update columns landing in the block, in child
      // order, at xrange[3 b ..], kb of them
      at.assign(y.chptr[s + 1] - y.chptr[s], 0);  // every child's first column not yet placed
      for (int j0 = 0; j0 < y.nrow[s]; j0 += 16) {
        FTask t{s, j0, (int)xrange.size() / 3, own(s), 0, 0};
        for (int q = y.chptr[s]; q < y.chptr[s + 1]; q++) {
          const int c = y.chlist[q], nu = y.nrow[c] - y.ncol[c];
          const int* rel = y.rel.data() + y.relptr[c];
          const int ka = at[q - y.chptr[s]];
          int kb = ka;
          while (kb < nu && rel[kb] < j0 + 16) kb++;
          at[q - y.chptr[s]] = kb;
          if (kb > ka) {
            xrange.push_back(c);
            xrange.push_back(ka);
            xrange.push_back(kb);
            t.kb++;
          }
        }
        tasks.push_back(t);
      }
    }
    if ((int)tasks.size() > off) ops.push_back({EXTADD, off, (int)tasks.size() - off, rows});
    int maxnc = 0;
    for (int q = 0; q < ns; q++) maxnc = std::max(maxnc, y.ncol[sups[q]]);
    // Pivot columns go in panels of up to P columns (sub-panels of 64): for
    // each sub-panel the diagonal block and the triangular solve, then its
    // update of the panel's remaining columns only; after the last sub-panel
    // one trailing update over the whole panel, so the trailing block is
    // read and written once per panel, and ceil(ncol / P) times per front
    // (factor of the 45x41x43 block: P = 64, 128, 192, 256 take 81, 62, 55,
    // 53 ms; of the 48x24x24 block 12.7, 11.4, 11.0, 11.0).
    // Panels with at most FUSE_TRSM row tiles below their diagonal blocks
    // (summed over the level) take one fused launch instead.
    constexpr int FUSE_TRSM = 256;
    auto add_diag_trsm = [&](int k0) {
      int ntr = 0;
      for (int q = 0; q < ns; q++) {
        int s = sups[q];
        if (y.ncol[s] > k0) ntr += (y.nrow[s] - k0 - std::min(64, y.ncol[s] - k0) + 63) / 64;
      }
      if (ntr <= FUSE_TRSM) {
        int off = (int)tasks.size();
        for (int q = 0; q < ns; q++) {
          int s = sups[q];
          if (y.ncol[s] <= k0) continue;
          int kb = std::min(64, y.ncol[s] - k0), rem = y.nrow[s] - k0 - kb;
          if (rem <= 0) tasks.push_back({s, -1, 0, k0, 0, 0});
          for (int a = 0; 64 * a < rem; a++) tasks.push_back({s, a, 0, k0, 0, 0});
        }
        if ((int)tasks.size() > off) ops.push_back({DIAG_TRSM, off, (int)tasks.size() - off});
        return;
      }
      int off = (int)tasks.size();
      for (int q = 0; q < ns; q++) {
        int s = sups[q];
        if (y.ncol[s] > k0) tasks.push_back({s, 0, 0, k0, 0, 0});
      }
      if ((int)tasks.size() > off) ops.push_back({DIAG, off, (int)tasks.size() - off});
      off = (int)tasks.size();
      for (int q = 0; q < ns; q++) {
        int s = sups[q];
        if (y.ncol[s] <= k0) continue;
        int kb = std::min(64, y.ncol[s] - k0), rem = y.nrow[s] - k0 - kb;
        for (int a = 0; 64 * a < rem; a++) tasks.push_back({s, a, 0, k0, 0, 0});
      }
      if ((int)tasks.size() > off) ops.push_back({TRSM, off, (int)tasks.size() - off});
    };
    // 64x64 lower tiles of the trailing block from k0 + kb, tile columns in
    // [tlo, thi) (thi < 0: all), columns before je (0: all), appended to `out`
    auto add_update_to = [&](std::vector<FTask>& out, int s, int k0, int kb, int tlo, int thi, int je) {
      const int rem = y.nrow[s] - k0 - kb;
      if (rem <= 0) return;
      const int T = (rem + 63) / 64;
      for (int ti = 0; ti < T; ti++)
        for (int tj = tlo; tj <= ti && (thi < 0 || tj < thi); tj++) out.push_back({s, ti, tj, k0, kb, je});
      // lower-triangle entries (incl. diagonal) of the updated columns c in
      // [clo, chi), rem - c each, 2 flops per FMA
      double clo = std::min(rem, 64 * tlo), chi = thi < 0 ? rem : std::min(rem, 64 * thi);
      if (je > 0) chi = std::min(chi, (double)(je - k0 - kb));
      if (chi > clo) flops += 2.0 * kb * ((chi - clo) * rem - (chi * (chi - 1) - clo * (clo - 1)) / 2);
    };
    const int P = panel, NA = P / 64;
    // Lookahead on the levels of few large fronts (those that take the fused
    // diagonal/TRSM launch): the trailing update after a panel is split into
    // the tiles of the next panel's columns (main stream) and the rest (side
    // stream), so the next panel's diagonal blocks, TRSM and narrow update
    // run while the rest of the trailing block is updated.  Any update that
    // reaches past the next panel joins the side stream first, and so does
    // the end of the level.
    int ntr0 = 0;
    for (int q = 0; q < ns; q++) {
      int s = sups[q];
      if (y.ncol[s] > 0) ntr0 += (y.nrow[s] - std::min(64, y.ncol[s]) + 63) / 64;
    }
    const bool look = lookahead && ntr0 <= FUSE_TRSM;
    bool side_pending = false;
    for (int k0 = 0; k0 < maxnc; k0 += P) {
      for (int h = 0; h < P / 64 && k0 + 64 * h < maxnc; h++) {
        const int kh = k0 + 64 * h;
        add_diag_trsm(kh);
        const int off = (int)tasks.size();
        std::vector<FTask> side;
        bool past = false;  // some task updates columns past the next panel
        for (int q = 0; q < ns; q++) {
          int s = sups[q];
          const int rc = y.ncol[s] - k0, w = std::min(P, rc);  // this front's panel
          if (rc <= 64 * h) continue;
          if (64 * (h + 1) < w) {  // the panel's remaining columns
            add_update_to(tasks, s, kh, 64, 0, (w - 64 * (h + 1) + 63) / 64, k0 + w);
          } else {  // the trailing block, whole panel
            if (look && rc > P) {
              add_update_to(tasks, s, k0, w, 0, NA, 0);
              add_update_to(side, s, k0, w, NA, -1, 0);
            } else {
              add_update_to(tasks, s, k0, w, 0, -1, 0);
            }
            past = true;
          }
        }
        if ((int)tasks.size() > off) {
          if (past && side_pending) {
            ops.push_back({JOIN, 0, 0});
            side_pending = false;
          }
          ops.push_back({UPDATE, off, (int)tasks.size() - off});
        }
        if (!side.empty()) {
          const int soff = (int)tasks.size();
          tasks.insert(tasks.end(), side.begin(), side.end());
          ops.push_back({FORK, 0, 0});
          ops.push_back({UPDATE_SIDE, soff, (int)side.size()});
          side_pending = true;
        }
      }
    }
    if (side_pending) ops.push_back({JOIN, 0, 0});
  }
  // Explicit inverse of every pivot block, joined pairwise from its diagonal
  // tiles (k_inv_mul).  Only the solves read the inverses, so they are formed
  // after the whole factorisation, over all fronts at once, long sums first.
  int maxT = 0;
  for (int s = 0; s < y.nsup; s++) maxT = std::max(maxT, (y.ncol[s] + 63) / 64);
  for (int h = 1; h < maxT; h *= 2) {
    std::vector<FTask> join[2];
    int at = 0;  // in 16-element units
    for (int s = 0; s < y.nsup; s++) {
      const int T = (y.ncol[s] + 63) / 64;
      for (int m = h; m < T; m += 2 * h) {
        const int end = std::min(m + h, T);
        for (int i = m; i < end; i++)
          for (int j = m - h; j < m; j++)
            for (int f = 0; f < 2; f++) join[f].push_back({s, j, i, 64 * m, f, at});
        at += 4 * h * (std::min(64 * (m + h), y.ncol[s]) - 64 * m);  // as inverse_products counts
      }
    }
    auto terms = [](const FTask& t) { return t.kb ? t.b - t.k0 / 64 + 1 : t.k0 / 64 - t.a; };
    for (auto& q : join) {
      std::stable_sort(q.begin(), q.end(), [&](const FTask& a, const FTask& b) { return terms(a) > terms(b); });
      ops.push_back({INV_MUL, (int)tasks.size(), (int)q.size()});
      tasks.insert(tasks.end(), q.begin(), q.end());
    }
  }
  // Y21 of the fused levels, long sums first
  std::vector<FTask> pan;
  for (int l = 0; l < y.nlevels; l++) {
    if (!lay.fused[l]) continue;
    for (int q = y.lvptr[l]; q < y.lvptr[l + 1]; q++) {
      const int s = y.lvsup[q], nu = y.nrow[s] - y.ncol[s];
      for (int j = 0; 64 * j < y.ncol[s]; j++)
        for (int i = 0; 64 * i < nu; i++) pan.push_back({s, j, i, y.ncol[s] - 64 * j, 0, 0});
    }
  }
  std::stable_sort(pan.begin(), pan.end(), [](const FTask& a, const FTask& b) { return a.k0 > b.k0; });
  if (!pan.empty()) {
    ops.push_back({PANEL, (int)tasks.size(), (int)pan.size()});
    tasks.insert(tasks.end(), pan.begin(), pan.end());
  }
}

// First work row of every front (nsup + 1 entries) and the gather lists of
// the forward init: work row woff[s] + i of front s adds the update rows of
// s's children that land in its row i, child after child (a child adds at
// most one row to a parent row).
static std::vector<int> work_rows(const Symbolic& y) {
  std::vector<int> woff(y.nsup + 1, 0);
  for (int s = 0; s < y.nsup; s++) woff[s + 1] = woff[s] + y.nrow[s];
  return woff;
}
static void build_gather(const Symbolic& y, std::vector<int>& gptr, std::vector<int>& gsrc, std::vector<int2>& kids) {
  const std::vector<int> woff = work_rows(y);
  gptr.assign(woff[y.nsup] + 1, 0);
  for (int s = 0; s < y.nsup; s++)
    for (int q = y.chptr[s]; q < y.chptr[s + 1]; q++) {
      const int c = y.chlist[q], nu = y.nrow[c] - y.ncol[c];
      const int* rel = y.rel.data() + y.relptr[c];
      for (int k = 0; k < nu; k++) gptr[woff[s] + rel[k] + 1]++;
    }
  for (size_t i = 1; i < gptr.size(); i++) gptr[i] += gptr[i - 1];
  gsrc.assign(std::max(1, gptr.back()), 0);
  std::vector<int> fill(gptr.begin(), gptr.end() - 1);
  for (int s = 0; s < y.nsup; s++)
    for (int q = y.chptr[s]; q < y.chptr[s + 1]; q++) {
      const int c = y.chlist[q], nu = y.nrow[c] - y.ncol[c];
      const int* rel = y.rel.data() + y.relptr[c];
      for (int k = 0; k < nu; k++) gsrc[fill[woff[s] + rel[k]]++] = woff[c] + y.ncol[c] + k;
    }
  kids.resize(std::max(1, woff[y.nsup]));
  for (int w = 0; w < woff[y.nsup]; w++) {
    const int n = gptr[w + 1] - gptr[w];
    kids[w] = int2{n > 0 ? gsrc[gptr[w]] : -1, n > 1 ? gsrc[gptr[w] + 1] : -1};
  }
}

// Solve plan for sp.nrhs right-hand sides: per level a forward init (fronts
// with children), one product in a fused level and two in another, then the
// levels top-down.  zero_start: also the backward pass from Y = 0.  Where no
// front of a level has more than two children (a separator that is empty or
// falls apart gives more), the products gather the update rows, and the pivot
// rows too in a level of few source bytes (GM_BYTES): the init is left with the
// pivot rows or with nothing.  A step of the 17x13x11 block's Lanczos loop is 8
// launches shorter (reduction 4.83 -> 4.65 ms), the inits of a forward pass of
// the 45x41x43 block take 70 us instead of 170.
//
// Right-hand sides go in groups of up to 96 columns, as even as 16-column
// tiles allow.  A task's K range is split over the 4 waves of a workgroup
// (the fastest split from 60 to 5544 pivot columns, see k_fw); over 16 (8
// for wide groups) where there is at most one 4-wave workgroup per CU and a
// wave would have more than ksplit of it; and not at all where it is short
// or, forward, where a level of short ranges (K <= ksplit) has enough rows
// to fill the device with 64-row tasks (24 against 28 us for 306 fronts of
// 700 rows and 60 pivot columns).
static void build_solve_plan(const Symbolic& y, const SolveLayout& lay, SolvePlan& sp, PlanHost& h, int ksplit,
                             bool zero_start) {
  const int nrhs = sp.nrhs, schur = y.nsup - 1;
  const int ngrp = (nrhs + 95) / 96;
  sp.nt = ((nrhs + ngrp - 1) / ngrp + 15) / 16;
  const std::vector<int> woff = work_rows(y);
  // rows of an init task: one value a thread, as each is a chain of three loads
  // (64 rows by 66 columns took four in turn: a launch 9.6 us, now 4.7)
  const int ir = std::max(4, std::min(64, 1024 / nrhs));
  // one launch: (task with its whole row range, rows) pieces, cut into row tiles
  struct Piece {
    MvTask t;      // rn = all rows
    int64_t da;    // operand step per target row
    int tri;       // 1: row tile r0 takes K up to r0 + rn (lower triangle), 2: K from r0 on, 0: all
  };
  auto cut = [&](std::vector<Op>& ops, int kind, const std::vector<Piece>& ps) {
    int64_t t16 = 0;
    int kmax = 0;
    for (const Piece& p : ps) {
      t16 += (p.t.rn + 15) / 16 * ngrp;
      kmax = std::max(kmax, p.t.kn);
    }
    const bool fw = kind == FW_MV || kind == FW_MV_ADD || kind == FW_MV_ALL;
    const bool wide = fw && t16 >= 4096 && kmax <= ksplit;
    Op op{kind, (int)h.tasks.size(), 0, 4};
    if (wide || kmax <= 32) op.kw = 1;
    else if (t16 <= 256 && kmax > 4 * ksplit) op.kw = 16;
    const int rt = op.kw == 1 && fw ? 64 : 16;
    for (const Piece& p : ps)
      for (int r0 = 0; r0 < p.t.rn; r0 += rt) {
        MvTask t = p.t;
        t.rn = std::min(rt, p.t.rn - r0);
        t.a += p.da * r0;
        t.dst += r0;
        if (t.dst2 >= 0) t.dst2 += r0;
        if (p.tri == 1) t.kn = std::min(t.kn, r0 + t.rn);
        if (p.tri == 2) {
          const int step = std::min(r0, t.kn);
          t.a += step;
          t.src += step;
          t.ky -= std::min(step, t.ky);
          t.kn -= step;
        }
        for (int g = 0; g < ngrp; g++) {
          t.j0 = 16 * sp.nt * g;
          if (t.j0 < nrhs) h.tasks.push_back(t);
        }
      }
    op.n = (int)h.tasks.size() - op.off;
    if (op.n > 0) ops.push_back(op);
  };
  for (int l = 0; l < y.nlevels; l++) {
    const int i0 = (int)h.inits.size();
    std::vector<Piece> first, second;
    bool pairs = l > 0;  // (the fronts of level 0 have no children)
    int64_t bytes = 0;
    for (int q = y.lvptr[l]; q < y.lvptr[l + 1]; q++) {
      const int s = y.lvsup[q];
      pairs = pairs && (s == schur || y.chptr[s + 1] - y.chptr[s] <= 2);
      bytes += (int64_t)((y.nrow[s] + 15) / 16) * y.ncol[s] * 128 * sp.nt * ngrp;
    }
    const bool all = pairs && sp.nt <= GM_TILES && bytes <= GM_BYTES;
    for (int q = y.lvptr[l]; q < y.lvptr[l + 1]; q++) {
      const int s = y.lvsup[q];
      if (s == schur) continue;
      const int nc = y.ncol[s], nu = y.nrow[s] - nc, ld = lay.ild[s];
      const bool leaf = y.chptr[s + 1] == y.chptr[s], up = y.parent[s] != schur && y.parent[s] >= 0;
      // rows that only the boundary would take are not formed
      const int rows = up && !pairs ? y.nrow[s] : nc;
      if (!leaf && !all)
        for (int r0 = 0; r0 < rows; r0 += ir)
          h.inits.push_back({woff[s] + r0, std::min(ir, rows - r0), std::max(0, std::min(ir, nc - r0)), y.col0[s] + r0});
      const int from = leaf ? y.col0[s] : woff[s], ff = leaf ? MV_SRC_R : 0;
      const size_t pieces = first.size();
      if (lay.fused[l]) {
        if (up)
          first.push_back({{lay.ioff[s] + nc, ld, nu, nc, from, 0, woff[s] + nc, -1, ff | (leaf ? MV_SET : MV_ADD), 0, 0}, 1, 0});
        first.push_back({{lay.ioff[s], ld, nc, nc, from, 0, y.col0[s], -1, ff | MV_Y, 0, 0}, 1, 1});
      } else {
        first.push_back({{lay.ioff[s], ld, nc, nc, from, 0, y.col0[s], up ? woff[s] : -1, ff | MV_Y, 0, 0}, 1, 1});
        if (up)
          second.push_back({{y.foff[s] + nc, y.nrow[s], nu, nc, woff[s], 0, woff[s] + nc, -1,
                             MV_FRONT | MV_SRC_V | (leaf ? MV_NEG : MV_SUB), 0, 0}, 1, 0});
      }
      for (size_t p = pieces; p < first.size(); p++) first[p].t.rsrc = y.col0[s];
    }
    if ((int)h.inits.size() > i0) sp.fw.push_back({FW_INIT, i0, (int)h.inits.size() - i0});
    cut(sp.fw, all ? FW_MV_ALL : pairs ? FW_MV_ADD : FW_MV, first);
    cut(sp.fw, pairs ? FW_MV_ADD : FW_MV, second);
  }
  for (int z = 0; z < (zero_start ? 2 : 1); z++) {
    std::vector<Op>& ops = z ? sp.bw0 : sp.bw;
    for (int l = y.nlevels - 1; l >= 0; l--) {
      std::vector<Piece> first, second;
      for (int q = y.lvptr[l]; q < y.lvptr[l + 1]; q++) {
        const int s = y.lvsup[q];
        if (s == schur) continue;
        const int nc = y.ncol[s], nu = y.nrow[s] - nc, ld = lay.ild[s];
        if (lay.fused[l]) {
          if (z)
            first.push_back({{lay.ioff[s] + nc, ld, nc, nu, y.rptr[s] + nc, 0, y.col0[s], -1, MV_X, 0, 0}, ld, 0});
          else
            first.push_back({{lay.ioff[s], ld, nc, nc + nu, y.rptr[s], nc, y.col0[s], -1, MV_X, 0, 0}, ld, 2});
        } else {
          first.push_back({{y.foff[s] + nc, y.nrow[s], nc, nu, y.rptr[s] + nc, 0, woff[s], y.col0[s],
                            MV_FRONT | MV_YSUB, 0, 0}, y.nrow[s], 0});
          second.push_back({{lay.ioff[s], ld, nc, nc, woff[s], 0, y.col0[s], -1, MV_X, 0, 0}, ld, 2});
        }
      }
      cut(ops, BW_ROWS, first);
      cut(ops, BW_MV, second);
    }
  }
}

int DeviceReducer::analyze(const Part& p, const ReduceOptions& o, std::string& err, bool upload_now) {
  const auto t0 = std::chrono::steady_clock::now();
  part_ = p;
  opt_ = o;
  if (build_sam(part_, sam_, err)) return -1;
  // inputReducerModule.f90:403-409: NGEN may not exceed NDOF1; the number of
  // eigenpairs is at most NDOF1
  if (opt_.ngen > sam_.ndof1) {
    err = "The number of generalized DOFs (NGEN) is larger than the number of internal nodal DOFs (NDOF1): "
          "NGEN = " + std::to_string(opt_.ngen) + ", NDOF1 = " + std::to_string(sam_.ndof1) +
          ". Reduce NGEN to less than NDOF1.";
    return -1;
  }
  opt_.neval = std::min(opt_.neval, sam_.ndof1);
  if (build_symbolic(part_, sam_, opt_.sym, sym_, err)) return -1;
  d_->hexl.clear();
  d_->shl.clear();
  d_->bml.clear();
  for (int e = 0; e < part_.nel; e++) {
    if (part_.etype[e] == HEX8) d_->hexl.push_back(e);
    else if (part_.etype[e] == ANDES4) d_->shl.push_back(e);
    else if (part_.etype[e] == BEAM2) d_->bml.push_back(e);
    else {
      err = "element type " + std::to_string(part_.etype[e]) + " not supported on the device path yet";
      return -2;
    }
  }
  uploaded_ = false;
  times_.analyze_host = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  // upload_now with a device: the upload (and the device structure build and
  // the solve plans) happens here, on the caller's thread, so that a caller
  // that analyses the next part while another handle reduces overlaps all of
  // it; otherwise it waits for the first reduce()
  if (!upload_now) return 0;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) == hipSuccess && ndev > 0) return upload(err);
  (void)hipGetLastError();
  return 0;
}

// The lookahead side stream and its events, created only for a schedule that
// forks (an idle extra stream per reducer would share the hardware queues
// with the streams of other reducers).
static hipError_t ensure_side(DeviceReducer::Impl& d) {
  bool fork = false;
  for (const Op& op : d.fops) fork = fork || op.kind == FORK;
  if (!fork || d.side) return hipSuccess;
  hipError_t e = hipStreamCreateWithFlags(&d.side, hipStreamNonBlocking);
  for (auto& ev : d.fj)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  return e;
}

// The assembled-matrix structure built on the device from the host's
// ordering and fronts: CSR columns, the pull-assembly contribution lists
// (in a fixed order) and the front map (structure.hip).  Checks the
// contribution count against the host's and reports entries outside the
// pattern.
int DeviceReducer::build_structure(std::string& err) {
  Impl& d = *d_;
  const Symbolic& y = sym_;
  const int nnz = y.rowptr[y.neq];
  HIPCHK(d.madof.upload(sam_.madof));
  HIPCHK(d.msc.upload(sam_.msc));
  HIPCHK(d.nndof.upload(sam_.nndof));
  HIPCHK(d.ceq_ptr.upload(sam_.ceq_ptr));
  HIPCHK(d.ceq_node.upload(sam_.ceq_node));
  HIPCHK(d.ceq_dof.upload(sam_.ceq_dof));
  HIPCHK(d.ceq_coef.upload(sam_.ceq_coef));
  HIPCHK(d.drank.upload(y.drank));
  HIPCHK(d.etype.upload(part_.etype));
  HIPCHK(d.nfirst.upload(y.nfirst));
  HIPCHK(d.neqd.upload(y.neqd));
  HIPCHK(d.nbptr.upload(y.nbptr));
  HIPCHK(d.nbl.upload(y.nbl));
  HIPCHK(d.rnode.upload(y.rnode));
  HIPCHK(d.colsn.upload(y.colsn));
  HIPCHK(d.rowptr.upload(y.rowptr));
  HIPCHK(d.row0.upload(y.nrow0));
  d.nnode = (int)y.nrow0.size() - 1;
  HIPCHK(d.nbo.alloc(std::max<size_t>(1, y.nbl.size())));
  HIPCHK(d.colind.alloc(nnz));
  HIPCHK(d.cptr.alloc((size_t)nnz + 1));
  HIPCHK(d.cidx.alloc(y.ncontrib));
  if (y.has_rigid) HIPCHK(d.ccoef.alloc(y.ncontrib));
  else d.ccoef.release();
  HIPCHK(d.fmap.alloc(nnz));
  HIPCHK(d.dpos.alloc(y.neq));
  DBuf<int>&cnt = d.sb_cnt, &tsum = d.sb_tsum, &bad = d.sb_bad;
  HIPCHK(cnt.alloc((size_t)nnz));
  HIPCHK(tsum.alloc((size_t)scan_tiles(nnz) + 1));
  HIPCHK(bad.alloc(1));
  HIPCHK(d.hpiv.alloc(PIVOT_STATS));
  hipStream_t st = st_;
  HIPCHK(d.batch.flush());
  HIPCHK(hipMemsetAsync(bad.p, 0, sizeof(int), st));
  launch_nbr_sort(st, part_.nnod, d.nbptr.p, d.nbl.p, d.nfirst.p, d.neqd.p, d.nbo.p);
  launch_csr_cols(st, y.neq, d.rnode.p, d.rowptr.p, d.nbptr.p, d.nbl.p, d.nbo.p, d.nfirst.p, d.neqd.p, d.colind.p);
  double* ccoef = y.has_rigid ? d.ccoef.p : nullptr;
  for (int pass = 0; pass < 2; pass++) {
    HIPCHK(hipMemsetAsync(cnt.p, 0, sizeof(int) * (size_t)nnz, st));
    launch_contrib(st, pass, part_.nel, d.etype.p, d.eptr.p, d.enodes.p, d.eoff.p, d.madof.p, d.msc.p, d.nndof.p,
                   d.ceq_ptr.p, d.ceq_node.p, d.ceq_dof.p, d.ceq_coef.p, d.drank.p, d.nfirst.p, d.rowptr.p, d.nbptr.p,
                   d.nbl.p, d.nbo.p, cnt.p, d.cptr.p, d.cidx.p, ccoef, bad.p);
    if (pass == 0) launch_exclusive_scan(st, nnz, cnt.p, d.cptr.p, tsum.p);
  }
  launch_seg_sort(st, nnz, d.cptr.p, d.cidx.p, ccoef);
  launch_fmap(st, y.neq, d.rowptr.p, d.colind.p, d.colsn.p, d.S, d.fmap.p, d.dpos.p, bad.p);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(d.hpiv.p, bad.p, sizeof(int), hipMemcpyDeviceToHost, st));
  HIPCHK(hipMemcpyAsync(d.hpiv.p + 1, d.cptr.p + nnz, sizeof(int), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  d.stage.passed();
  const int hb = d.hpiv.p[0], total = d.hpiv.p[1];
  if (hb || total != y.ncontrib) {
    err = "device structure build: " + std::string(hb & 1 ? "element contribution outside the CSR pattern" :
                                                   hb & 2 ? "matrix entry outside its front" :
                                                            "contribution count mismatch");
    return -3;
  }
  return 0;
}

// Device upload of the part and of every structure array the kernels read.
static void lanczos_sizes(int n1, int nev, const ReduceOptions& o, int& bs, int& mcap);
static SolvePlan* plan_slot(DeviceReducer::Impl& d, int nrhs);
static void plan_host(const Symbolic& y, const DeviceReducer::Impl& d, SolvePlan& sp, PlanHost& h);
static int plan_upload(SolvePlan& sp, const PlanHost& h, std::string& err);

int DeviceReducer::upload(std::string& err) {
  const auto t0 = std::chrono::steady_clock::now();
  // FGPU_TRACE_REDUCE=1: host-side timeline of the upload on stderr
  const bool trace = std::getenv("FGPU_TRACE_REDUCE") != nullptr;
  auto mark = [&](const char* what) {
    if (trace)
      std::fprintf(stderr, "upload +%.2f ms: %s\n",
                   std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count(), what);
  };
  Impl& d = *d_;
  if (!st_) {
    // non-blocking: no implicit ordering with the null stream (and so with
    // other threads' null-stream copies); default priority
    HIPCHK(hipStreamCreateWithFlags(&st_, hipStreamNonBlocking));
    for (auto& e : d.ev) HIPCHK(hipEventCreate(&e));
  }
  StreamScope scope(st_);
  HIPCHK(d.batch.open(st_));
  BatchScope gather(d.batch);
  HIPCHK(d.xyz.upload(part_.xyz));
  HIPCHK(d.eprop.upload(part_.eprop));
  HIPCHK(d.eptr.upload(part_.eptr));
  HIPCHK(d.enodes.upload(part_.enodes));
  HIPCHK(d.hexlist.upload(d.hexl));
  {
    std::vector<int> p1(sym_.ndof1);  // permuted row of every internal equation, in MEQN1 order
    for (int q = 0; q < sym_.ndof1; q++) p1[q] = sym_.eq_to_perm[sam_.meqn1[q] - 1];
    HIPCHK(d.p1.upload(p1));
  }
  HIPCHK(d.shlist.upload(d.shl));
  HIPCHK(d.bmlist.upload(d.bml));
  HIPCHK(d.eoff.upload(sym_.elem_off));
  mark("part arrays");
  const Symbolic& y = sym_;
  HIPCHK(d.col0.upload(y.col0));
  HIPCHK(d.ncol.upload(y.ncol));
  HIPCHK(d.nrow.upload(y.nrow));
  HIPCHK(d.rptr.upload(y.rptr));
  HIPCHK(d.rows.upload(y.rows));
  HIPCHK(d.chptr.upload(y.chptr));
  HIPCHK(d.chlist.upload(y.chlist));
  HIPCHK(d.relptr.upload(y.relptr));
  HIPCHK(d.rel.upload(y.rel));
  HIPCHK(d.foff.upload(y.foff));
  d.wrows = work_rows(y)[y.nsup];
  d.lay = solve_layout(y, opt_);
  const std::vector<int64_t>& ioff = d.lay.ioff;
  HIPCHK(d.ioff.upload(ioff));
  HIPCHK(d.ild.upload(d.lay.ild));
  d.mixed = opt_.mixed;
  d.m_diag = d.hexl.empty() && d.bml.empty() && !y.has_rigid;
  d.solve_split = std::max(64, (opt_.solve_split / 64) * 64);
  if (d.mixed) {
    d.ipool.release();
    HIPCHK(d.ipool32.alloc(ioff[y.nsup] + PANEL_PAD));
  } else {
    d.ipool32.release();
    HIPCHK(d.ipool.alloc(ioff[y.nsup] + PANEL_PAD));
  }
  HIPCHK(d.dpiv.alloc((size_t)std::max(1, y.ndof1)));
  HIPCHK(d.adiag.alloc((size_t)std::max(1, y.ndof1)));
  HIPCHK(d.amax.alloc(1));
  HIPCHK(d.sing.alloc((size_t)std::max(1, y.ndof1)));
  d.S = DevSym{d.col0.p, d.ncol.p, d.nrow.p, d.foff.p, d.rptr.p, d.rows.p, d.chptr.p,
               d.chlist.p, d.relptr.p, d.rel.p, d.ild.p, d.dpiv.p,
               d.adiag.p, d.amax.p, d.sing.p, std::max(opt_.tol_factorize, 1e-20)};
  // The host-side schedules (the factorisation's and the solve plans the
  // reduction uses) are built on host threads while the device builds the
  // structure.  The solve plans keep their device buffers: freeing them
  // would wait for the whole device.
  for (auto& kv : d.plans) kv.second->valid = false;
  std::vector<int> want;
  {
    const int n1 = y.ndof1, n2 = y.ndof2;
    const int nev = opt_.ngen > 0 ? std::max(opt_.neval, opt_.ngen) : 0;
    if (n1 > 0 && n2 > 0) want.push_back(n2);
    if (n1 > 0 && nev > 0) {
      int bs = 0, mcap = 0;
      lanczos_sizes(n1, nev, opt_, bs, mcap);
      if (std::find(want.begin(), want.end(), bs) == want.end()) want.push_back(bs);
    }
    if (n1 > 0 && opt_.want_vgi && std::find(want.begin(), want.end(), 3) == want.end()) want.push_back(3);
  }
  std::vector<SolvePlan*> sps;
  for (int nr : want) sps.push_back(plan_slot(d, nr));
  std::vector<PlanHost> phs(sps.size());
  std::vector<FTask> ft;
  d.fops.clear();
  std::vector<int> xr;
  const int panel = opt_.factor_panel == ReduceOptions::PANEL_DEFAULT
                        ? (opt_.mixed ? 64 : 256)
                        : std::min(256, std::max(64, (opt_.factor_panel / 64) * 64));
  std::vector<int> gptr, gsrc;
  std::vector<int2> kids;
  HostJobs host_jobs;  // (after all that the jobs write)
  host_jobs.start([&]() {
    build_factor_schedule(y, d.lay, ft, d.fops, xr, upd_flops_, panel, opt_.factor_lookahead);
  });
  host_jobs.start([&]() { build_gather(y, gptr, gsrc, kids); });
  for (size_t i = 0; i < sps.size(); i++) host_jobs.start([&, i]() { plan_host(y, d, *sps[i], phs[i]); });
  const int src = build_structure(err);
  host_jobs.wait();
  if (src) return src;
  mark("structure built");
  HIPCHK(d.gptr.upload(gptr));
  HIPCHK(d.gsrc.upload(gsrc));
  HIPCHK(d.kids.upload(kids));
  for (size_t i = 0; i < sps.size(); i++)
    if (int rc = plan_upload(*sps[i], phs[i], err)) return rc;
    else sps[i]->valid = true;
  HIPCHK(ensure_side(d));
  HIPCHK(d.ftasks.upload(ft));
  mark("factor schedule built");
  HIPCHK(d.xrange.upload(xr));
  HIPCHK(d.itmp.alloc((size_t)inverse_workspace(y) + PANEL_PAD));
  upd_launches_ = 0;
  for (auto& op : d.fops)
    if (op.kind == UPDATE || op.kind == UPDATE_SIDE) upd_launches_++;
  // a new structure: every captured launch sequence is stale
  d.g_factor.reset();
  d.factor_runs = 0;
  // value buffers
  const int64_t nnz = y.rowptr[y.neq];
  HIPCHK(d.Kp.alloc(y.elem_pool));
  HIPCHK(d.Mp.alloc(y.elem_pool));
  HIPCHK(d.Kv.alloc(nnz));
  HIPCHK(d.Mv.alloc(nnz));
  if (d.mixed) {
    d.pool.release();
    HIPCHK(d.pool32.alloc(y.fpool + PANEL_PAD));
    HIPCHK(d.dscale.alloc(y.neq));
    HIPCHK(d.dcs.alloc(std::max(1, y.ndof2)));
    HIPCHK(d.irpart.alloc(2 * SUMSQ_BLOCKS));
  } else {
    d.pool32.release();
    HIPCHK(d.pool.alloc(y.fpool + PANEL_PAD));
  }
  HIPCHK(d.ebad.alloc(part_.nel));
  HIPCHK(d.emass.alloc(part_.nel + 1));
  HIPCHK(d.piv.alloc(PIVOT_STATS));
  mark("value buffers");
  // gravity directions: unit accelerations on translational equation DOFs
  std::vector<double> a((size_t)y.neq * 3, 0.0);
  for (int i = 0; i < sam_.nnod; i++)
    for (int j = 0; j < 3 && j < sam_.nndof[i]; j++) {
      int dof = sam_.madof[i] - 1 + j;
      if (sam_.meqn[dof] > 0) a[(size_t)y.eq_to_perm[sam_.meqn[dof] - 1] * 3 + j] = 1.0;
    }
  HIPCHK(d.grav.upload(a));
  HIPCHK(d.e2p.upload(y.eq_to_perm));
  HIPCHK(d.pos2.upload(sam_.dofPosIn2.empty() ? std::vector<int>(1, 1) : sam_.dofPosIn2));
  mark("gravity and maps");
  // the solve plans and work buffers the reduction will use, made here (on
  // the caller's analysis thread) instead of on the reduction's path
  if (int rc = prepare_solves(err)) return rc;
  HIPCHK(d.batch.flush());
  mark("solve plans");
  uploaded_ = true;
  times_.upload = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return 0;
}

// The slot of the plan for nrhs right-hand sides: the existing plan (its
// device buffers reused, its host lists cleared) or a new one in the map.
static SolvePlan* plan_slot(DeviceReducer::Impl& d, int nrhs) {
  auto it = d.plans.find(nrhs);
  SolvePlan* sp = nullptr;
  if (it != d.plans.end()) {
    sp = it->second.get();
    sp->fw.clear();
    sp->bw.clear();
    sp->bw0.clear();
  } else {
    auto fresh = std::make_unique<SolvePlan>();
    sp = fresh.get();
    d.plans[nrhs] = std::move(fresh);
  }
  sp->valid = false;
  sp->nrhs = nrhs;
  return sp;
}

// Host part of a plan (pure host work, safe on another thread).  B has as
// many right-hand sides as boundary equations, so their plan gets the
// backward pass from zero too.
static void plan_host(const Symbolic& y, const DeviceReducer::Impl& d, SolvePlan& sp, PlanHost& h) {
  build_solve_plan(y, d.lay, sp, h, d.solve_split, sp.nrhs == y.ndof2);
}

static int plan_upload(SolvePlan& sp, const PlanHost& h, std::string& err) {
  HIPCHK(sp.tasks.upload(h.tasks));
  HIPCHK(sp.inits.upload(h.inits));
  return 0;
}

static int get_plan(const Symbolic& y, DeviceReducer::Impl& d, int nrhs, SolvePlan*& out, std::string& err) {
  auto it = d.plans.find(nrhs);
  if (it != d.plans.end() && it->second->valid) { out = it->second.get(); return 0; }
  SolvePlan* sp = plan_slot(d, nrhs);
  PlanHost h;
  plan_host(y, d, *sp, h);
  if (tl_batch) {
    if (int rc = plan_upload(*sp, h, err)) return rc;
  } else {  // a plan made for a call after the upload
    HIPCHK(d.batch.open(tl_stream));
    BatchScope gather(d.batch);
    if (int rc = plan_upload(*sp, h, err)) return rc;
    HIPCHK(d.batch.flush());
  }
  sp->valid = true;
  out = sp;
  return 0;
}

static int ensure_work(DeviceReducer::Impl& d, int nrhs, std::string& err) {
  HIPCHK(d.W.alloc((size_t)d.wrows * nrhs));
  if (d.lay.unfused) HIPCHK(d.V.alloc((size_t)d.wrows * nrhs));
  return 0;
}

// Lanczos block size and basis capacity for nev modes of n1 internal
// equations: blocks of lanczos_block vectors (<= 64, the Gram matrices' limit),
// lanczosMaxVectors or max(10 nev + 40, 16 blocks) vectors, at least nev, in
// whole blocks; a basis that would span the whole internal space takes a
// block size dividing n1, so that it does so exactly.
static void lanczos_sizes(int n1, int nev, const ReduceOptions& o, int& bs, int& mcap) {
  bs = std::max(1, std::min(std::min(o.lanczos_block, 64), n1));
  mcap = o.lanczos_maxvec > 0 ? o.lanczos_maxvec : std::max(10 * nev + 40, 16 * bs);
  mcap = (std::max(mcap, nev) + bs - 1) / bs * bs;
  if (mcap >= n1) {
    while (n1 % bs) bs--;
    mcap = n1;
  }
}

int DeviceReducer::prepare_solves(std::string& err) {
  Impl& d = *d_;
  const Symbolic& y = sym_;
  const int n1 = y.ndof1, n2 = y.ndof2, neq = y.neq;
  const int nev = opt_.ngen > 0 ? std::max(opt_.neval, opt_.ngen) : 0;
  if (n1 <= 0) return 0;
  SolvePlan* p = nullptr;
  if (n2 > 0) {
    if (get_plan(y, d, n2, p, err)) return -3;
    if (ensure_work(d, n2, err)) return -3;
    HIPCHK(d.X.alloc((size_t)neq * n2));
    HIPCHK(d.Z.alloc((size_t)neq * n2));
    HIPCHK(d.Y.alloc((size_t)neq * n2));
  }
  if (nev > 0) {
    int bs = 0, mcap = 0;
    lanczos_sizes(n1, nev, opt_, bs, mcap);
    if (get_plan(y, d, bs, p, err)) return -3;
    if (ensure_work(d, std::max(bs, n2), err)) return -3;
    HIPCHK(d.Q.alloc((size_t)neq * mcap));
    HIPCHK(d.P.alloc((size_t)neq * mcap));
    HIPCHK(d.Wl.alloc((size_t)neq * bs));
    HIPCHK(d.Zl.alloc((size_t)neq * bs));
    HIPCHK(d.Yl.alloc((size_t)neq * bs));
    HIPCHK(d.Tmp.alloc((size_t)neq * bs));
    HIPCHK(d.Cc.alloc((size_t)mcap * std::max(bs, nev) + 64));
    HIPCHK(d.part.alloc((size_t)xty_chunks(neq) * mcap * std::max(bs, nev)));
    HIPCHK(d.small.alloc((size_t)mcap * mcap + 64));
    HIPCHK(d.lzrec.alloc(1 + (size_t)2 * bs * bs + (size_t)mcap * bs));
    HIPCHK(d.signs.alloc((size_t)nev * (1 + 3 * MODE_SIGN_GROUPS)));
  }
  if (opt_.want_vgi && get_plan(y, d, 3, p, err)) return -3;
  return 0;
}

static void run_mv(hipStream_t st, DeviceReducer::Impl& d, const SolvePlan& sp, const Op& op, const double* R,
                   double* Y, double* X) {
  const MvTask* t = sp.tasks.p + op.off;
  const int kind = op.kind == FW_MV ? MV_FORWARD : op.kind == FW_MV_ADD ? MV_FORWARD_ADD :
                   op.kind == FW_MV_ALL ? MV_FORWARD_ALL : op.kind == BW_ROWS ? MV_BACK_ROWS : MV_BACK;
  if (d.mixed)
    launch_mv(st, t, op.n, kind, sp.nt, op.kw, d.pool32.p, d.ipool32.p, d.S.rows, d.S.dpiv, d.kids.p, d.W.p, d.V.p, R, Y,
              X, sp.nrhs);
  else
    launch_mv(st, t, op.n, kind, sp.nt, op.kw, d.pool.p, d.ipool.p, d.S.rows, d.S.dpiv, d.kids.p, d.W.p, d.V.p, R, Y, X,
              sp.nrhs);
}

// Z = M X
static void mass_mm(hipStream_t st, int neq, const DeviceReducer::Impl& d, int nrhs, const double* X, int ldx, double* Z,
                    int ldz) {
  if (d.m_diag) launch_diag_mm(st, neq, nrhs, d.dpos.p, d.Mv.p, X, ldx, Z, ldz);
  else launch_spmm(st, d.node_rows(neq), nrhs, d.rowptr.p, d.colind.p, d.Mv.p, X, ldx, Z, ldz);
}

// Y = D^{-1} L^{-1} R on the internal rows
static void run_forward(hipStream_t st, DeviceReducer::Impl& d, const SolvePlan& sp, const double* R, double* Y) {
  for (const Op& op : sp.fw) {
    if (op.kind == FW_INIT)
      launch_fw_init(st, sp.inits.p + op.off, op.n, d.gptr.p, d.gsrc.p, R, d.W.p, sp.nrhs);
    else
      run_mv(st, d, sp, op, R, Y, nullptr);
  }
}

// X = L^{-T} Y on the internal rows (Y null: zero); X's boundary rows must
// be set by the caller
static void run_backward(hipStream_t st, DeviceReducer::Impl& d, const SolvePlan& sp, double* Y, double* X) {
  for (const Op& op : Y ? sp.bw : sp.bw0) run_mv(st, d, sp, op, nullptr, Y, X);
}

// Relative size ||D|| / ||X|| of a correction D against the solution X
// over their first n entries (device partial sums, added in block order).
static int rel_correction(hipStream_t st, DeviceReducer::Impl& d, int64_t n, const double* D, const double* X,
                          double& rel, std::string& err) {
  launch_sumsq2(st, n, D, X, d.irpart.p);
  double h[2 * SUMSQ_BLOCKS];
  HIPCHK(hipMemcpyAsync(h, d.irpart.p, sizeof h, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  double a = 0.0, b = 0.0;
  for (int q = 0; q < SUMSQ_BLOCKS; q++) {
    a += h[2 * q];
    b += h[2 * q + 1];
  }
  rel = b > 0.0 ? std::sqrt(a / b) : (a > 0.0 ? INFINITY : 0.0);
  return 0;
}

// Stopping rule of the mixed-precision refinement, from the relative size of
// the latest correction: done when it is below tol, or when it no longer
// halves (the residual has reached FP64 rounding level, where the
// correction is noise of the size cond(K) * eps64); failure when it stays
// large past the step limit, or above 0.1 after 12 steps.
static int refine_state(double rel, double prev, int steps, const ReduceOptions& opt, std::string& err,
                        const char* what) {
  if (rel <= opt.ir_tol) return 1;
  if (steps >= 2 && rel > 0.5 * prev && rel < 1e-6) return 1;
  // a correction still above 0.1 after 12 steps has contracted by less than
  // 0.83 a step: it cannot reach ir_tol within the step limit, so stop now
  if (steps >= opt.ir_maxit || !std::isfinite(rel) || (steps >= 12 && rel > 0.1)) {
    char buf[160];
    std::snprintf(buf, sizeof buf, "mixed-precision iterative refinement of %s did not converge "
                  "(correction %.3e after %d steps)", what, rel, steps);
    err = buf;
    return -1;
  }
  return 0;
}

// One approximate solve D = K_ii^{-1} R on the mixed-precision factor:
// D = S (K~_ii)^{-1} S R with K~ = S K S the equilibrated matrix whose FP32
// LDL^T the fronts hold.  R's internal rows are read, `scaled` takes S R (neq x
// nrhs); D's boundary rows are zero.
static void approx_solve(hipStream_t st, DeviceReducer::Impl& d, const SolvePlan& sp, int neq, int ndof1,
                         const double* R, double* scaled, double* Yw, double* D) {
  launch_scale_rc(st, ndof1, sp.nrhs, d.dscale.p, nullptr, R, scaled);
  run_forward(st, d, sp, scaled, Yw);
  launch_fill(st, D + (size_t)ndof1 * sp.nrhs, (int64_t)(neq - ndof1) * sp.nrhs, 0.0);  // boundary rows
  run_backward(st, d, sp, Yw, D);
  launch_scale_rc(st, ndof1, sp.nrhs, d.dscale.p, nullptr, D, D);
}

// Mixed precision: conjugate gradients on K_ii X = b, one independent CG
// per column, preconditioned by the FP32 factor (z = K~_ii^-1 r through
// approx_solve), residuals and updates in FP64.  The stationary refinement
// X += K~^-1 r contracts each step by the spread rho of the preconditioned
// spectrum about 1; CG by about rho / (1 + sqrt(1 - rho^2)) and faster
// where the spectrum clusters.  On entry X holds the starting solution and
// R (neq x nr, internal rows) its residual b - K_ii X; X's boundary rows
// are left alone.  A column whose curvature p^T K_ii p or r^T z is not
// positive (an indefinite K_ii or factor) turns the remaining steps into
// stationary refinement for all columns.  Stopping: refine_state on the
// relative size of the step's correction.
static int pcg_int(hipStream_t st, DeviceReducer::Impl& d, const Symbolic& y, const ReduceOptions& opt,
                   const SolvePlan& sp, double* X, double* R, double* Yw, int* steps, const char* what,
                   std::string& err) {
  const int neq = y.neq, n1 = y.ndof1, nr = sp.nrhs;
  const int64_t nall = (int64_t)neq * nr, nint = (int64_t)n1 * nr;
  HIPCHK(d.cg_p.alloc(nall));
  HIPCHK(d.cg_q.alloc(nall));
  HIPCHK(d.cg_z.alloc(nall));
  HIPCHK(d.cg_t.alloc(nall));
  HIPCHK(d.cg_part.alloc((size_t)std::max(1, coldot_blocks(n1)) * 3 * nr));
  HIPCHK(d.cg_dot.alloc((size_t)3 * nr));
  HIPCHK(d.cg_co.alloc((size_t)3 * nr));
  std::vector<double> h((size_t)3 * nr), rz(nr), xx(nr), co((size_t)3 * nr);
  // column dot products of npair pairs over the internal rows, to h
  auto dots = [&](int npair, const double* A0, const double* B0, const double* A1, const double* B1,
                  const double* A2, const double* B2) -> int {
    launch_coldots(st, n1, nr, npair, A0, B0, A1, B1, A2, B2, d.cg_part.p, d.cg_dot.p);
    HIPCHK(hipMemcpyAsync(h.data(), d.cg_dot.p, sizeof(double) * npair * nr, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return 0;
  };
  // z = K~^-1 r
  auto precond = [&]() { approx_solve(st, d, sp, neq, n1, R, d.cg_t.p, Yw, d.cg_z.p); };
  bool stationary = false;
  double prev = INFINITY;
  precond();
  if (int rc = dots(2, R, d.cg_z.p, X, X, nullptr, nullptr)) return rc;
  for (int c = 0; c < nr; c++) {
    rz[c] = h[c];
    xx[c] = h[nr + c];  // |X_c|^2, carried through the updates for the stopping rule
    if (!(rz[c] >= 0.0)) stationary = true;
  }
  // p = z (boundary rows zero, so K p has K_ii p in its internal rows)
  HIPCHK(hipMemcpyAsync(d.cg_p.p, d.cg_z.p, sizeof(double) * nall, hipMemcpyDeviceToDevice, st));
  for (int it = 0;; it++) {
    double rel = 0.0;
    if (stationary) {
      // X += z; r = b - K_ii X = r - K_ii z
      launch_axpby(st, nint, 1.0, d.cg_z.p, 1.0, X);
      launch_spmm(st, d.node_rows(neq), nr, d.rowptr.p, d.colind.p, d.Kv.p, d.cg_z.p, nr, d.cg_q.p, nr);
      launch_axpby(st, nint, -1.0, d.cg_q.p, 1.0, R);
      if (rel_correction(st, d, nint, d.cg_z.p, X, rel, err)) return -3;
    } else {
      launch_spmm(st, d.node_rows(neq), nr, d.rowptr.p, d.colind.p, d.Kv.p, d.cg_p.p, nr, d.cg_q.p, nr);
      if (int rc = dots(3, d.cg_p.p, d.cg_q.p, d.cg_p.p, d.cg_p.p, d.cg_p.p, X)) return rc;
      double num = 0.0, den = 0.0;
      for (int c = 0; c < nr; c++) {
        const double pq = h[c], pp = h[nr + c], px = h[2 * nr + c];
        double a = 0.0;
        if (rz[c] > 0.0) {
          if (pq > 0.0) a = rz[c] / pq;
          else stationary = true;
        }
        co[c] = a;
        co[nr + c] = -a;
        num += a * a * pp;
        xx[c] += a * (2.0 * px + a * pp);  // |X_c + a p_c|^2
        den += xx[c];
      }
      if (stationary) {  // fall back from the current X and r: redo this step as a stationary one
        it--;
        continue;
      }
      HIPCHK(hipMemcpyAsync(d.cg_co.p, co.data(), sizeof(double) * 2 * nr, hipMemcpyHostToDevice, st));
      launch_col_axpby(st, n1, nr, d.cg_co.p, d.cg_p.p, nullptr, X);           // X += a p
      launch_col_axpby(st, n1, nr, d.cg_co.p + nr, d.cg_q.p, nullptr, R);      // r -= a K p
      rel = den > 0.0 ? std::sqrt(num / den) : (num > 0.0 ? INFINITY : 0.0);
    }
    if (steps) *steps = it + 1;
    if (std::getenv("FGPU_TRACE_REFINE"))  // FGPU_TRACE_REFINE=1: each step's correction on stderr
      std::fprintf(stderr, "refine %s step %d: |dX|/|X| %.3e%s\n", what, it + 1, rel,
                   stationary ? " (stationary)" : "");
    const int state = refine_state(rel, prev, it + 1, opt, err, what);
    if (state > 0) return 0;
    if (state < 0) return -6;
    prev = rel;
    precond();
    if (stationary) continue;
    if (int rc = dots(1, R, d.cg_z.p, nullptr, nullptr, nullptr, nullptr)) return rc;
    for (int c = 0; c < nr; c++) {
      const double rzn = h[c];
      if (!(rzn >= 0.0)) stationary = true;
      co[2 * nr + c] = rz[c] > 0.0 ? rzn / rz[c] : 0.0;
      rz[c] = rzn;
    }
    if (stationary) continue;
    HIPCHK(hipMemcpyAsync(d.cg_co.p + 2 * nr, co.data() + 2 * nr, sizeof(double) * nr, hipMemcpyHostToDevice, st));
    launch_col_axpby(st, n1, nr, nullptr, d.cg_z.p, d.cg_co.p + 2 * nr, d.cg_p.p);  // p = z + beta p
  }
}

// X = K_ii^{-1} R on the internal rows (X's boundary rows zero), R and X
// neq x nrhs row-major in perm order; Yw is neq x nrhs work.  FP64 factor:
// one forward and one backward pass.  Mixed precision: conjugate gradients
// preconditioned by the FP32 factor with residuals from the FP64 CSR
// matrix (pcg_int), until the correction is below ir_tol relative to X.
static int solve_int(hipStream_t st, DeviceReducer::Impl& d, const Symbolic& y, const ReduceOptions& opt,
                     const SolvePlan& sp, const double* R, double* Yw, double* X, int* steps, std::string& err) {
  const int neq = y.neq, n1 = y.ndof1, nr = sp.nrhs;
  const int64_t nall = (int64_t)neq * nr, nint = (int64_t)n1 * nr;
  if (!d.mixed) {
    run_forward(st, d, sp, R, Yw);
    launch_fill(st, X + nint, nall - nint, 0.0);  // boundary rows; the backward pass writes the others
    run_backward(st, d, sp, Yw, X);
    if (steps) *steps = 0;
    return 0;
  }
  // conjugate gradients from X = 0 (residual R)
  HIPCHK(d.Rr.alloc(nall));
  HIPCHK(hipMemcpyAsync(d.Rr.p, R, sizeof(double) * nall, hipMemcpyDeviceToDevice, st));
  launch_fill(st, X, nall, 0.0);
  return pcg_int(st, d, y, opt, sp, X, d.Rr.p, Yw, steps, "a K_ii solve", err);
}

static double ev_ms(hipEvent_t a, hipEvent_t b) {
  float ms = 0;
  (void)hipEventElapsedTime(&ms, a, b);
  return ms;
}

int DeviceReducer::reduce(std::string& err) {
  if (!uploaded_) {
    int rc = upload(err);
    if (rc) return rc;
  }
  StreamScope scope(st_);
  // FGPU_TRACE_REDUCE=1: host-side timeline of the phases on stderr
  const bool trace = std::getenv("FGPU_TRACE_REDUCE") != nullptr;
  const auto tr0 = std::chrono::steady_clock::now();
  auto mark = [&](const char* what) {
    if (trace)
      std::fprintf(stderr, "reduce +%.2f ms: %s\n",
                   std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tr0).count(), what);
  };
  Impl& d = *d_;
  const Symbolic& y = sym_;
  const int neq = y.neq, n1 = y.ndof1, n2 = y.ndof2, schur = y.nsup - 1;
  const int64_t nnz = y.rowptr[neq];
  const int nev = opt_.ngen > 0 ? std::max(opt_.neval, opt_.ngen) : 0;
  const int ngen = opt_.ngen;
  hipStream_t st = st_;
  res_ = Results();
  times_.refine_steps = 0;
  res_.ndof1 = n1;
  res_.ndof2 = n2;
  res_.ngen = ngen;
  res_.nev = nev;
  res_.ndim = sam_.ndim_ext + ngen;
  HIPCHK(hipEventRecord(d.ev[0], st));
  mark("start issued");
  // ---- element matrices
  launch_begin(st, part_.nel, d.ebad.p, std::max(1, n1), d.sing.p, d.piv.p, d.amax.p);
  launch_hex8(st, (int)d.hexl.size(), d.hexlist.p, d.eptr.p, d.enodes.p, d.xyz.p, d.eprop.p, d.eoff.p, d.Kp.p,
              d.Mp.p, d.ebad.p);
  launch_andes4(st, (int)d.shl.size(), d.shlist.p, d.eptr.p, d.enodes.p, d.xyz.p, d.eprop.p, d.eoff.p, d.Kp.p,
                d.Mp.p, d.ebad.p);
  launch_beam(st, (int)d.bml.size(), d.bmlist.p, d.eptr.p, d.enodes.p, d.xyz.p, d.eprop.p, d.eoff.p, d.Kp.p,
              d.Mp.p, d.ebad.p);
  if (!opt_.no_mass) {  // total FE mass (SMASS of lhsINADD) for the reduced-mass check
    launch_emass(st, (int)d.hexl.size(), d.hexlist.p, 8, 3, d.eoff.p, d.Mp.p, d.emass.p);
    launch_emass(st, (int)d.shl.size(), d.shlist.p, 4, 6, d.eoff.p, d.Mp.p, d.emass.p);
    launch_emass(st, (int)d.bml.size(), d.bmlist.p, 2, 6, d.eoff.p, d.Mp.p, d.emass.p);
    launch_sum_fixed(st, part_.nel, d.emass.p, d.emass.p + part_.nel);
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(d.ev[1], st));
  // ---- assembly (CSR K, M and the K entries of the fronts)
  const Op& fz = d.fops.front();
  if (d.mixed) launch_front_zero(st, d.ftasks.p + fz.off, fz.n, d.S, d.pool32.p);
  else launch_front_zero(st, d.ftasks.p + fz.off, fz.n, d.S, d.pool.p);
  launch_assemble(st, nnz, d.cptr.p, d.cidx.p, y.has_rigid ? d.ccoef.p : nullptr, d.Kp.p, d.Mp.p, d.Kv.p, d.Mv.p,
                  d.fmap.p, d.mixed ? nullptr : d.pool.p);
  if (d.mixed) {  // equilibrated stiffness into the FP32 fronts
    launch_diag_scale(st, neq, d.dpos.p, d.Kv.p, d.dscale.p);
    launch_front_scatter32(st, neq, d.rowptr.p, d.colind.p, d.Kv.p, d.dscale.p, d.fmap.p, d.pool32.p);
  }
  // original diagonal of K_ii for the singular-pivot test (equilibrated for
  // the mixed-precision factor), no pivot flagged yet
  launch_diag_extract(st, n1, d.dpos.p, d.Kv.p, d.mixed ? d.dscale.p : nullptr, d.adiag.p, d.amax.p);
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(d.ev[2], st));
  mark("elements and assembly issued");
  // ---- multifrontal LDL^T; the Schur front ends up holding K_bb - K_bi K_ii^-1 K_ib
  if (opt_.time_updates && d.upd_ev.size() < 2 * (size_t)upd_launches_) {  // another schedule may launch more
    const size_t have = d.upd_ev.size();
    d.upd_ev.resize(2 * (size_t)upd_launches_);
    for (size_t q = have; q < d.upd_ev.size(); q++) HIPCHK(hipEventCreate(&d.upd_ev[q]));
  }
  int64_t ui = 0;
  hipError_t fork_err = hipSuccess;  // first failure of a fork or join of the side stream
  auto note = [&](hipError_t e) {
    if (e != hipSuccess && fork_err == hipSuccess) fork_err = e;
  };
  auto factor_with = [&](auto* pool, auto* ipool) {
    for (const Op& op : d.fops) {
      switch (op.kind) {
        case EXTADD: launch_extend_add(st, d.ftasks.p + op.off, op.n, op.kw, d.S, d.xrange.p, pool); break;
        case DIAG: launch_diag(st, d.ftasks.p + op.off, op.n, d.S, pool, d.ioff.p, ipool); break;
        case TRSM: launch_trsm(st, d.ftasks.p + op.off, op.n, d.S, pool, d.ioff.p, ipool); break;
        case DIAG_TRSM: launch_diag_trsm(st, d.ftasks.p + op.off, op.n, d.S, pool, d.ioff.p, ipool); break;
        case UPDATE:
        case UPDATE_SIDE: {
          // with per-launch timing everything stays on the main stream
          hipStream_t us = (op.kind == UPDATE_SIDE && !opt_.time_updates) ? d.side : st;
          if (opt_.time_updates) (void)hipEventRecord(d.upd_ev[2 * ui], st);
          launch_update(us, d.ftasks.p + op.off, op.n, d.S, pool);
          if (opt_.time_updates) (void)hipEventRecord(d.upd_ev[2 * ui + 1], st);
          ui++;
          break;
        }
        case FORK:
          if (!opt_.time_updates) {
            note(hipEventRecord(d.fj[0], st));
            note(hipStreamWaitEvent(d.side, d.fj[0], 0));
          }
          break;
        case JOIN:
          if (!opt_.time_updates) {
            note(hipEventRecord(d.fj[1], d.side));
            note(hipStreamWaitEvent(st, d.fj[1], 0));
          }
          break;
        case INV_MUL:
          launch_inv_mul(st, d.ftasks.p + op.off, op.n, d.S, pool, d.ioff.p, ipool,
                         reinterpret_cast<decltype(pool)>(d.itmp.p));
          break;
        case PANEL: launch_panel(st, d.ftasks.p + op.off, op.n, d.S, pool, d.ioff.p, ipool); break;
      }
    }
  };
  auto factor_ops = [&]() {
    if (d.mixed) factor_with(d.pool32.p, d.ipool32.p);
    else factor_with(d.pool.p, d.ipool.p);
  };
  // The first factorisation after an upload runs eagerly (a part reduced
  // once gains nothing from a capture); later ones replay one captured graph.
  if (opt_.time_updates || !opt_.use_graphs || d.factor_runs++ == 0) {
    factor_ops();  // per-launch events need the plain stream
  } else {
    // the factor schedule is fixed per symbolic structure: one graph
    HIPCHK(run_graph(st, d.g_factor,
                     {d.ftasks.p, d.xrange.p, d.itmp.p, d.pool.p, d.ipool.p, d.pool32.p, d.ipool32.p, d.ioff.p,
                      d.S.foff, d.S.rows, d.S.dpiv},
                     factor_ops));
  }
  HIPCHK(fork_err);
  launch_pivot_stats(st, n1, d.dpiv.p, d.sing.p, part_.nel, d.ebad.p, d.piv.p);
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(d.ev[3], st));
  mark("factor issued");
  // ---- B = -K_ii^{-1} K_ib: back-substitution of [0; I].  With the FP64
  // factor and component modes it is queued after the Lanczos steps instead,
  // where it runs on the device while the host solves the final projected
  // eigenproblem (events 8 and 9 bracket it there).
  SolvePlan* pb = nullptr;
  const bool defer_b = n2 > 0 && !d.mixed && nev > 0;
  if (n2 > 0) {
    if (get_plan(y, d, n2, pb, err)) return -3;
    if (ensure_work(d, n2, err)) return -3;
    HIPCHK(d.X.alloc((size_t)neq * n2));
    HIPCHK(d.Z.alloc((size_t)neq * n2));
    HIPCHK(d.Y.alloc((size_t)neq * n2));
  }
  // the deferred pass also forms the mass phase's Z = M [B; I] (events 9-11)
  const bool defer_z = defer_b && !opt_.no_mass;
  auto issue_bsolve = [&]() -> int {
    HIPCHK(hipEventRecord(d.ev[8], st));
    launch_identity_rows(st, d.X.p + (size_t)n1 * n2, neq - n1, n2, 0);  // the backward pass writes rows < n1
    run_backward(st, d, *pb, nullptr, d.X.p);
    HIPCHK(hipEventRecord(d.ev[9], st));
    if (defer_z) {
      mass_mm(st, neq, d, n2, d.X.p, n2, d.Z.p, n2);
      HIPCHK(hipEventRecord(d.ev[11], st));
    }
    return 0;
  };
  if (n2 > 0 && !defer_b) {
    launch_identity_rows(st, d.X.p + (size_t)n1 * n2, neq - n1, n2, 0);  // the backward pass writes rows < n1
    run_backward(st, d, *pb, nullptr, d.X.p);
    if (d.mixed) {
      // the backward pass of the equilibrated factor gives S_i^-1 B S_b
      launch_recip(st, n2, d.dscale.p + n1, d.dcs.p);
      launch_scale_rc(st, n1, n2, d.dscale.p, d.dcs.p, d.X.p, d.X.p);
      // refinement against the FP64 matrix: Z = K [B; I] has the residual
      // -(K_ii B + K_ib) in its internal rows and K_bb + K_bi B in its
      // boundary rows (the Schur complement once B has converged)
      // conjugate gradients on K_ii B = -K_ib from this B: the internal
      // rows of K [B; I] are -(the residual), its boundary rows K_bb + K_bi B
      // (the Schur complement once B has converged)
      launch_spmm(st, d.node_rows(neq), n2, d.rowptr.p, d.colind.p, d.Kv.p, d.X.p, n2, d.Z.p, n2);
      launch_axpby(st, (int64_t)n1 * n2, -1.0, d.Z.p, 0.0, d.Z.p);
      int steps = 0;
      if (int rc = pcg_int(st, d, y, opt_, *pb, d.X.p, d.Z.p, d.Y.p, &steps, "B", err)) return rc;
      launch_spmm(st, d.node_rows(neq), n2, d.rowptr.p, d.colind.p, d.Kv.p, d.X.p, n2, d.Z.p, n2);
      times_.refine_steps = steps;
      std::vector<double> zb((size_t)n2 * n2);
      HIPCHK(hipMemcpyAsync(zb.data(), d.Z.p + (size_t)n1 * n2, sizeof(double) * zb.size(), hipMemcpyDeviceToHost,
                            st));
      HIPCHK(hipStreamSynchronize(st));
      d.s22.assign((size_t)n2 * n2, 0.0);
      for (int b = 0; b < n2; b++)
        for (int a = 0; a < n2; a++) d.s22[a + (size_t)b * n2] = 0.5 * (zb[(size_t)a * n2 + b] + zb[(size_t)b * n2 + a]);
    }
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(d.ev[4], st));
  mark("B issued");
  // error checks of the numeric phase
  HIPCHK(d.hpiv.alloc(PIVOT_STATS));
  HIPCHK(hipMemcpyAsync(d.hpiv.p, d.piv.p, sizeof(int) * PIVOT_STATS, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  d.stage.passed();
  int hbad[PIVOT_STATS];
  std::copy(d.hpiv.p, d.hpiv.p + PIVOT_STATS, hbad);
  if (const int e = hbad[6]; e != INT_MAX) {
    int code = 0;
    HIPCHK(d2h(&code, d.ebad.p + e, sizeof code));
    err = "element " + std::to_string(e + 1) +
          (code == -3 ? " has a degenerate shell geometry (zero area or length)"
                      : " has a non-positive Jacobian determinant");
    return -4;
  }
  res_.n_negative = hbad[0];
  res_.n_true_zero = hbad[1];
  res_.n_reduced_zero = hbad[2];
  if (hbad[1] + hbad[2] > 0) {
    std::vector<int> sg(n1);
    HIPCHK(hipMemcpyAsync(sg.data(), d.sing.p, sizeof(int) * n1, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    for (int c = 0; c < n1; c++)
      if (sg[c]) res_.singular.push_back({y.perm_to_eq[c], sg[c]});
    std::sort(res_.singular.begin(), res_.singular.end());
    const int h = opt_.sing_handler;
    const bool abort = h == 0 || (h == 1 && hbad[2] > 0);
    if (abort) {
      const int c = h == 0 ? std::min(hbad[4], hbad[5]) : hbad[5];
      err = "singular K_ii: " + std::to_string(hbad[1]) + " zero and " + std::to_string(hbad[2]) +
            " reduced-to-zero pivot(s) (tolFactorize " + std::to_string(opt_.tol_factorize) + ", singularityHandler " +
            std::to_string(h) + "); first at equation " + std::to_string(y.perm_to_eq[c] + 1);
      return -5;
    }
  }
  // ---- component modes (block Lanczos, shift-invert on the resident factor)
  if (nev > 0) {
    int rc = 0;
    int bs = 0, mcap = 0;
    lanczos_sizes(n1, nev, opt_, bs, mcap);
    SolvePlan* pl = nullptr;
    if (get_plan(y, d, bs, pl, err)) return -3;
    if (ensure_work(d, std::max(bs, n2), err)) return -3;
    HIPCHK(d.Q.alloc((size_t)neq * mcap));
    HIPCHK(d.P.alloc((size_t)neq * mcap));
    HIPCHK(d.Wl.alloc((size_t)neq * bs));
    HIPCHK(d.Zl.alloc((size_t)neq * bs));
    HIPCHK(d.Yl.alloc((size_t)neq * bs));
    HIPCHK(d.Tmp.alloc((size_t)neq * bs));
    HIPCHK(d.Cc.alloc((size_t)mcap * std::max(bs, nev) + 64));
    HIPCHK(d.part.alloc((size_t)xty_chunks(neq) * mcap * std::max(bs, nev)));
    HIPCHK(d.small.alloc((size_t)mcap * mcap + 64));
    const size_t nrec = 1 + (size_t)2 * bs * bs, slot = nrec + (size_t)mcap * bs;
    HIPCHK(d.lzrec.alloc(slot));
    HIPCHK(d.hrec.alloc(2 * slot));
    double *const Rdev = d.lzrec.p + 1, *const Cacc = d.lzrec.p + nrec;
    int* const lzbad = reinterpret_cast<int*>(d.lzrec.p);
    for (auto& e : d.lz_ev)
      if (!e) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    // start block: pseudo-random values on the internal rows, zero boundary
    // rows, which every step leaves alone
    launch_start_block(st, neq, n1, bs, opt_.seed, d.Wl.p);
    std::vector<double> H((size_t)mcap * mcap, 0.0);
    // Block M-orthonormalisation of W (CholQR twice): G = W^T M W = R^T R on
    // the device, W <- W R^-1, M W <- (M W) R^-1, then Q_j = W and P_j = M W
    // (also in Tmp, the next solve's right-hand side).  orth_issue queues the
    // work, copy_rec the copy of the step's record with its first nc
    // coefficients to host slot `par`; orth_finish (after the stream has
    // passed it) forms R_tot = R_2 R_1, W = Q_j R_tot.
    auto orth_issue = [&](int j) {
      // M W is formed once: the second pass's M (W R_1^-1) is (M W) R_1^-1
      mass_mm(st, neq, d, bs, d.Wl.p, bs, d.Zl.p, bs);
      for (int pass = 0; pass < 2; pass++) {
        launch_gram_inv(st, neq, bs, d.Wl.p, d.Zl.p, d.part.p, d.Cc.p, Rdev + (size_t)pass * bs * bs, d.small.p,
                        pass == 0, lzbad);
        // the first pass rescales in place, the second writes block j
        if (pass == 0) launch_gemm_small2(st, neq, bs, bs, d.Wl.p, bs, d.Wl.p, bs, d.Zl.p, bs, d.Zl.p, bs, d.small.p);
        else
          launch_gemm_small2(st, neq, bs, bs, d.Wl.p, bs, d.Q.p + (size_t)j * bs, mcap, d.Zl.p, bs,
                             d.P.p + (size_t)j * bs, mcap, d.small.p, d.Tmp.p, bs);
      }
    };
    auto copy_rec = [&](int par, size_t nc) {
      return hipMemcpyAsync(d.hrec.p + par * slot, d.lzrec.p, sizeof(double) * (nrec + nc), hipMemcpyDeviceToHost, st);
    };
    auto orth_finish = [&](int par, std::vector<double>& Rtot) -> int {
      if (*reinterpret_cast<const int*>(d.hrec.p + par * slot)) {
        err = "Lanczos: block breakdown (Gram matrix not positive definite)";
        return -6;
      }
      const double* R1 = d.hrec.p + par * slot + 1;
      const double* R2 = R1 + (size_t)bs * bs;
      Rtot.assign((size_t)bs * bs, 0.0);
      for (int a = 0; a < bs; a++)
        for (int b = 0; b < bs; b++) {
          double s = 0;
          for (int k = 0; k < bs; k++) s += R2[(size_t)a * bs + k] * R1[(size_t)k * bs + b];
          Rtot[(size_t)a * bs + b] = s;
        }
      return 0;
    };
    std::vector<double> R0;
    orth_issue(0);
    HIPCHK(copy_rec(0, 0));
    HIPCHK(hipStreamSynchronize(st));
    if ((rc = orth_finish(0, R0))) return rc;
    int nb = 0;  // number of completed blocks in H
    bool conv = false;
    // symmetrised block-tridiagonal projection of the first mj Lanczos vectors
    auto projected = [&](int mj) {
      std::vector<double> Hs((size_t)mj * mj);
      for (int a = 0; a < mj; a++)
        for (int b = 0; b < mj; b++) {
          double h1 = H[(size_t)a * mcap + b], h2 = H[(size_t)b * mcap + a];
          Hs[(size_t)a * mj + b] = (a <= b + bs && b <= a + bs) ? 0.5 * (h1 + h2) : 0.0;
        }
      return Hs;
    };
    // Ritz pairs of the projection and their relative residuals
    // ||R_{j+1} s_last|| / |theta| (theta = 1 / (lambda - shift))
    struct Check {
      int mj = 0;
      bool ok = false;
      double worst = 0.0;
      std::vector<double> w, V;
    };
    const double tol = opt_.tol_eig;
    // G = the M-Gram matrix of the next (unnormalised) Lanczos block: the
    // residual of Ritz vector s is sqrt(s_last^T G s_last)
    std::atomic<bool> stop{false};  // the outcome of the checks still running is not needed
    auto run_check = [bs, nev, tol, &stop](int mj, std::vector<double> Hs, std::vector<double> G) {
      Check c;
      c.mj = mj;
      if (!sym_eig_top(mj, Hs, nev, c.w, c.V, &stop)) return c;  // V column i: i-th largest theta
      c.ok = true;
      for (int i = 0; i < nev; i++) {
        double th = c.w[mj - 1 - i], r2 = 0.0;
        const double* v = &c.V[(size_t)(mj - bs) * nev + i];
        for (int a = 0; a < bs; a++) {
          double s = 0;
          for (int b = 0; b < bs; b++) s += G[(size_t)a * bs + b] * v[(size_t)b * nev];
          r2 += v[(size_t)a * nev] * s;
        }
        double rel = std::sqrt(std::max(r2, 0.0)) / std::fabs(th);
        c.worst = std::max(c.worst, rel);
        if (!(rel <= tol)) c.ok = false;
      }
      return c;
    };
    auto gram_of = [&](const std::vector<double>& Rm) {  // R^T R
      std::vector<double> Gm((size_t)bs * bs, 0.0);
      for (int a = 0; a < bs; a++)
        for (int b = 0; b < bs; b++) {
          double s = 0.0;
          for (int k = 0; k < bs; k++) s += Rm[(size_t)k * bs + a] * Rm[(size_t)k * bs + b];
          Gm[(size_t)a * bs + b] = s;
        }
      return Gm;
    };
    // Convergence tests on the projected problem run on host threads while the
    // device computes the next blocks: one for every second block from the
    // first that can hold the modes, at most CHECKS at a time.  The first in
    // their order that passes decides the basis whatever the timing, so every
    // result bit, and whether there is a result, depends on the data only;
    // blocks computed meanwhile are dropped.  (A test takes 0.9 ms at 176 vectors, six steps of a small part,
    // which waited for it two steps later.)
    constexpr size_t CHECKS = 3;
    struct Pending {
      int step;
      std::future<Check> f;
    };
    std::deque<Pending> pending;
    int next_check = 0;
    double worst = 0.0, decay = 1.0;  // of the tests so far
    Check done;
    struct StopChecks {
      std::atomic<bool>& s;
      ~StopChecks() { s = true; }
    } stop_checks{stop};
    // takes the outcomes in order while one is there, waiting for those of
    // tests started up to block `upto`; true once one has passed
    auto collect = [&](int upto) {
      while (!conv && !pending.empty()) {
        Pending& q = pending.front();
        if (q.step > upto && q.f.wait_for(std::chrono::seconds(0)) != std::future_status::ready) break;
        Check c = q.f.get();
        pending.pop_front();
        if (std::getenv("FGPU_TRACE_LANCZOS"))
          std::fprintf(stderr, "lanczos: check of %d vectors, worst %.2e\n", c.mj, c.worst);
        decay = worst > 0.0 ? c.worst / worst : 1.0;
        worst = c.worst;
        if (c.ok) {
          done = std::move(c);
          conv = true;
        }
      }
      return conv;
    };
    // The residual falls by at least the last factor from test to test: where
    // that puts a running test inside the tolerance, its outcome is waited for
    // before another block is issued (17x13x11 block 5.34 against 5.48 ms,
    // beam frame of 450 elements 3.75 / 3.87).
    auto expected = [&]() {
      double r = worst;
      for (auto& q : pending) {
        r *= decay;
        if (0.0 < r && r <= tol) return q.step;
      }
      return -1;
    };
    // Step j (device): W = K_ii^{-1} (M Q_j), two passes of full
    // reorthogonalisation against Q_0..Q_j (coefficients added up on the
    // device and copied to host slot j % 2), then the next block Q_{j+1}.
    // Steps are queued one ahead of the host's bookkeeping, so the device
    // never waits for the host between blocks.
    auto issue_step = [&](int j) -> int {
      const int mj = (j + 1) * bs, par = j & 1;
      if (d.mixed) {
        if (int rc2 = solve_int(st, d, y, opt_, *pl, d.Tmp.p, d.Yl.p, d.Wl.p, nullptr, err)) return rc2;
      } else {
        // launch by launch: a captured graph of the two passes costs more to
        // start and to join than it saves (17x13x11 block 5.61 against 5.50 ms,
        // 450-element frame 4.40 / 4.30, 48x24x24 block 66.4 / 66.0)
        run_forward(st, d, *pl, d.Tmp.p, d.Yl.p);
        run_backward(st, d, *pl, d.Yl.p, d.Wl.p);
      }
      for (int pass = 0; pass < 2; pass++) {
        // coefficients of the pass into Cc, their running sum into Cacc
        launch_xty(st, neq, mj, bs, d.P.p, mcap, d.Wl.p, bs, d.part.p, d.Cc.p, Cacc, pass > 0);
        launch_gemm_small(st, neq, mj, bs, d.Q.p, mcap, d.Cc.p, d.Wl.p, bs, 1.0, -1.0);
      }
      if (mj + bs <= mcap) orth_issue(j + 1);
      HIPCHK(copy_rec(par, (size_t)mj * bs));
      HIPCHK(hipEventRecord(d.lz_ev[par], st));
      return 0;
    };
    if ((rc = issue_step(0))) return rc;
    for (int j = 0; (j + 1) * bs <= mcap; j++) {
      const int mj = (j + 1) * bs, par = j & 1;
      const bool last = mj + bs > mcap;
      if (collect(-1) || collect(expected())) break;
      // a block that cannot be made (breakdown, refinement that does not
      // converge) is an error only if no test of the blocks before it passes:
      // which of them have been started depends on j alone, and all of them
      // are waited for
      auto ended = [&]() {
        if (rc == -6 && collect(INT_MAX)) err.clear();
        return conv;
      };
      if (!last && (rc = issue_step(j + 1))) {
        if (ended()) break;
        return rc;
      }
      HIPCHK(hipEventSynchronize(d.lz_ev[par]));
      const double* hc = d.hrec.p + par * slot + nrec;
      for (int a = 0; a < mj; a++)
        for (int b = 0; b < bs; b++) H[(size_t)a * mcap + j * bs + b] = hc[(size_t)a * bs + b];
      nb = j + 1;
      if (last) break;
      std::vector<double> Rn;
      if ((rc = orth_finish(par, Rn))) {
        if (ended()) break;
        return rc;
      }
      for (int a = 0; a < bs; a++)
        for (int b = 0; b < bs; b++) H[(size_t)(mj + a) * mcap + j * bs + b] = Rn[(size_t)a * bs + b];
      if (collect(-1)) break;
      if (j >= next_check && mj >= std::max(2 * nev, 3 * bs)) {
        if (pending.size() == CHECKS && collect(pending.front().step)) break;
        pending.push_back({j, std::async(std::launch::async, run_check, mj, projected(mj), gram_of(Rn))});
        next_check = j + 2;
      }
    }
    collect(nb);
    stop = conv;
    // without a converged test the Ritz pairs come from the full basis; the
    // M-Gram matrix of the last (reorthogonalised) block gives their residuals
    if (!conv) {
      mass_mm(st, neq, d, bs, d.Wl.p, bs, d.Zl.p, bs);
      launch_xty(st, neq, bs, bs, d.Wl.p, bs, d.Zl.p, bs, d.part.p, d.Cc.p);
      std::vector<double> Gl((size_t)bs * bs);
      HIPCHK(hipMemcpyAsync(Gl.data(), d.Cc.p, sizeof(double) * bs * bs, hipMemcpyDeviceToHost, st));
      HIPCHK(hipEventRecord(d.ev[10], st));
      if (defer_b && (rc = issue_bsolve())) return rc;
      HIPCHK(hipEventSynchronize(d.ev[10]));
      const auto tw = std::chrono::steady_clock::now();
      done = run_check(nb * bs, projected(nb * bs), Gl);
      if (std::getenv("FGPU_TRACE_LANCZOS"))
        std::fprintf(stderr, "lanczos: final check of %d vectors on the host took %.3f ms, worst %.2e\n", done.mj,
                     std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tw).count(),
                     done.worst);
    } else if (defer_b && (rc = issue_bsolve())) {
      return rc;
    }
    res_.lanczos_resid = done.worst;
    if (!done.ok) {
      char buf[200];
      std::snprintf(buf, sizeof buf, "component modes did not converge: worst relative Ritz residual %.3e after %d "
                    "Lanczos vectors (tolerance %.1e; raise lanczosMaxVectors)", done.worst, done.mj, tol);
      err = buf;
      return -7;
    }
    const int m = done.mj;
    std::vector<double> w, V;
    w.swap(done.w);
    V.swap(done.V);
    (void)conv;
    res_.lanczos_vectors = m;
    // Ritz vectors for the nev largest theta (lowest lambda), lambda ascending
    std::vector<double> S((size_t)m * nev);
    res_.lambda.resize(nev);
    res_.eval.resize(nev);
    for (int i = 0; i < nev; i++) {
      double lam = 1.0 / w[m - 1 - i] + opt_.eig_shift;
      res_.lambda[i] = lam;
      res_.eval[i] = lam < 0 ? -std::sqrt(-lam) : std::sqrt(lam);
      for (int a = 0; a < m; a++) S[(size_t)a * nev + i] = V[(size_t)a * nev + i];
    }
    HIPCHK(hipMemcpyAsync(d.small.p, S.data(), sizeof(double) * S.size(), hipMemcpyHostToDevice, st));
    HIPCHK(d.Phi.alloc((size_t)neq * nev));
    launch_gemm_small(st, neq, m, nev, d.Q.p, mcap, d.small.p, d.Phi.p, nev, 0.0, 1.0);
    // sign convention: the largest-magnitude component of every mode is positive
    HIPCHK(d.signs.alloc((size_t)nev * (1 + 3 * MODE_SIGN_GROUPS)));
    launch_mode_signs(st, n1, d.p1.p, d.Phi.p, neq, nev, d.signs.p);
  }
  HIPCHK(hipEventRecord(d.ev[5], st));
  mark("modes done on host");
  // ---- reduced mass: Z = M [B; I], M22 = [B; I]^T Z ; modes: K11, M11, M12
  const int nd = res_.ndim;
  const int maxab = std::max(std::max(n2, 3), std::max(nev, 1));
  const size_t nrec = 2 * (size_t)nd * nd + 3 * (size_t)nd + 1;  // SK, SM, G, element mass
  HIPCHK(d.part.alloc((size_t)xty_chunks(neq) * maxab * maxab));
  HIPCHK(d.acc.alloc(nrec + (size_t)n2 * n2 + 2 * (size_t)ngen * ngen + (size_t)ngen * n2 + 3 * (size_t)(n2 + ngen)));
  HIPCHK(d.hred.alloc(nrec));
  ReducedParts rp{};
  {
    double* at = d.acc.p + nrec;
    auto take = [&](size_t n) {
      double* r = at;
      at += n;
      return r;
    };
    rp.M22 = take((size_t)n2 * n2);
    rp.K11 = take((size_t)ngen * ngen);
    rp.M11 = take((size_t)ngen * ngen);
    rp.M12 = take((size_t)ngen * n2);
    rp.Ge = take(3 * (size_t)n2);
    rp.Gg = take(3 * (size_t)ngen);
  }
  auto xty = [&](int na, int nb, const double* X, int ldx, const double* Yv, int ldy, double* out, bool sym = false) {
    if (na > 0 && nb > 0) launch_xty(st, neq, na, nb, X, ldx, Yv, ldy, d.part.p, out, nullptr, false, sym);
  };
  if (!opt_.no_mass && n2 > 0) {
    if (!defer_z) mass_mm(st, neq, d, n2, d.X.p, n2, d.Z.p, n2);
    xty(n2, n2, d.X.p, n2, d.Z.p, n2, rp.M22, true);
  }
  if (ngen > 0) {
    HIPCHK(d.Yl.alloc((size_t)neq * std::max(ngen, opt_.lanczos_block)));
    launch_spmm(st, d.node_rows(neq), ngen, d.rowptr.p, d.colind.p, d.Kv.p, d.Phi.p, nev, d.Yl.p, ngen);
    xty(ngen, ngen, d.Phi.p, nev, d.Yl.p, ngen, rp.K11, true);
    if (!opt_.no_mass) {
      mass_mm(st, neq, d, ngen, d.Phi.p, nev, d.Yl.p, ngen);
      xty(ngen, ngen, d.Phi.p, nev, d.Yl.p, ngen, rp.M11, true);
      xty(ngen, n2, d.Phi.p, nev, d.Z.p, n2, rp.M12);
    }
  }
  HIPCHK(hipEventRecord(d.ev[6], st));
  // ---- gravity: g = M a ; G_e = [B; I]^T g ; G_g = Phi^T g
  const bool vgi = !opt_.no_mass && opt_.want_vgi && n1 > 0;
  if (!opt_.no_mass) {
    HIPCHK(d.Tmp.alloc((size_t)neq * std::max(3, std::max(opt_.lanczos_block, nev))));
    mass_mm(st, neq, d, 3, d.grav.p, 3, d.Tmp.p, 3);
    xty(n2, 3, d.X.p, n2, d.Tmp.p, 3, rp.Ge);
    xty(ngen, 3, d.Phi.p, nev, d.Tmp.p, 3, rp.Gg);
    if (vgi) {
      SolvePlan* p3 = nullptr;
      if (get_plan(y, d, 3, p3, err)) return -3;
      if (ensure_work(d, std::max(std::max(n2, 3), opt_.lanczos_block), err)) return -3;
      HIPCHK(d.Zl.alloc((size_t)neq * std::max(3, opt_.lanczos_block)));
      HIPCHK(d.Wl.alloc((size_t)neq * std::max(3, opt_.lanczos_block)));
      if (int rc2 = solve_int(st, d, y, opt_, *p3, d.Tmp.p, d.Zl.p, d.Wl.p, nullptr, err)) return rc2;
      launch_rows_out(st, n1, 3, d.p1.p, d.Wl.p, 3, nullptr, 0, d.Zl.p, n1);  // MEQN1 order
    }
  }
  if (nd > 0) {
    const bool s22 = n2 > 0 && !d.mixed;  // the Schur complement in the root front
    launch_reduced(st, nd, n2, ngen, d.pos2.p, s22 ? d.pool.p + y.foff[schur] : nullptr, rp,
                   opt_.no_mass ? nullptr : d.emass.p + part_.nel, d.acc.p);
    HIPCHK(hipGetLastError());
  }
  HIPCHK(hipEventRecord(d.ev[7], st));
  mark("mass and gravity issued");
  if (nd > 0)
    HIPCHK(hipMemcpyAsync(d.hred.p, d.acc.p, sizeof(double) * (opt_.no_mass ? (size_t)nd * nd : nrec),
                          hipMemcpyDeviceToHost, st));
  else if (!opt_.no_mass)
    HIPCHK(hipMemcpyAsync(d.hred.p + nrec - 1, d.emass.p + part_.nel, sizeof(double), hipMemcpyDeviceToHost, st));
  if (vgi) {
    res_.vgi.resize((size_t)n1 * 3);
    HIPCHK(hipMemcpyAsync(res_.vgi.data(), d.Zl.p, sizeof(double) * res_.vgi.size(), hipMemcpyDeviceToHost, st));
  }
  HIPCHK(hipStreamSynchronize(st));
  mark("device done");
  times_.elements = ev_ms(d.ev[0], d.ev[1]);
  times_.assembly = ev_ms(d.ev[1], d.ev[2]);
  times_.factor = ev_ms(d.ev[2], d.ev[3]);
  times_.bsolve = defer_b ? ev_ms(d.ev[8], d.ev[9]) : ev_ms(d.ev[3], d.ev[4]);
  const double zms = defer_z ? ev_ms(d.ev[9], d.ev[11]) : 0.0;
  times_.modes = ev_ms(d.ev[4], d.ev[5]) - (defer_b ? times_.bsolve : 0.0) - zms;
  times_.mass = ev_ms(d.ev[5], d.ev[6]) + zms;
  times_.gravity = ev_ms(d.ev[6], d.ev[7]);
  times_.total = ev_ms(d.ev[0], d.ev[7]);
  times_.update_kernel_ms = 0;
  times_.update_launches = 0;
  if (opt_.time_updates) {
    for (int64_t q = 0; q < ui; q++) times_.update_kernel_ms += ev_ms(d.upd_ev[2 * q], d.upd_ev[2 * q + 1]);
    times_.update_launches = ui;
  }
  const size_t nn = (size_t)nd * nd;
  const double* h = d.hred.p;
  res_.SK.assign(h, h + nn);
  if (!opt_.no_mass) {
    res_.SM.assign(h + nn, h + 2 * nn);
    res_.G.assign(h + 2 * nn, h + 2 * nn + 3 * (size_t)nd);
    res_.mass_fe = h[nrec - 1];
  }
  if (d.mixed) {  // the Schur complement from the refined B
    const std::vector<int>& pos2 = sam_.dofPosIn2;
    for (int j = 0; j < n2; j++)
      for (int i = 0; i < n2; i++) {
        const int a = pos2[i] - 1, b = pos2[j] - 1;
        res_.SK[i + (size_t)j * nd] = d.s22[std::max(a, b) + (size_t)std::min(a, b) * n2];
      }
  }
  return 0;
}

hipError_t DeviceReducer::d2h(void* dst, const void* src, size_t bytes) const {
  if (!st_) return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st_);
  return e == hipSuccess ? hipStreamSynchronize(st_) : e;
}

// The parts of a column-major n x nc array that go through a piece of the stage
// at a time: whole columns where one fits, else rows of up to 16 columns (the
// width of an ordering kernel's tile).
struct Pieces {
  int n, nc, rows, cols;
  Pieces(int n_, int nc_) : n(n_), nc(nc_) {
    const int most = Stage::PIECE / sizeof(double);
    cols = std::min(nc, std::max(16, most / std::max(1, n)));
    rows = std::min(n, most / std::max(1, cols));
  }
  // go(h, q0, m, c0, k): rows q0 .. q0 + m and columns c0 .. c0 + k, piece h
  template <class F>
  int each(F&& go) const {
    int h = 0;
    for (int c0 = 0; c0 < nc; c0 += cols)
      for (int q0 = 0; q0 < n; q0 += rows, h ^= 1)
        if (int rc = go(h, q0, std::min(rows, n - q0), c0, std::min(cols, nc - c0))) return rc;
    return 0;
  }
};

// copy(piece, array, doubles) for the contiguous runs of a part
template <class F>
static void runs(char* piece, double* array, int n, int q0, int m, int c0, int k, F&& copy) {
  double* p = reinterpret_cast<double*>(piece);
  array += q0 + (size_t)c0 * n;
  if (m == n) return copy(p, array, (size_t)m * k);
  for (int c = 0; c < k; c++) copy(p + (size_t)c * m, array + (size_t)c * n, (size_t)m);
}

// Rows map[0..n) of A + B (row-major, either may be null) to the host, column-
// major.  A kernel writes them in their order into a piece of the stage, and
// the host copies one piece out while the device fills the other: no device
// buffer, and the data crosses the bus once.  (With copies behind an ordering
// kernel into a buffer of its own, through the runtime's staging memory, B of a
// 16x12x10 block took 0.98 ms where the order on the host took 0.53; 0.2 now.)
int DeviceReducer::rows_to_host(int n, int nc, const int* map, const double* A, int lda, const double* B, int ldb,
                                double* out, std::string& err) const {
  Stage& s = d_->stage;
  HIPCHK(s.open());
  struct {
    int q0, m = 0, c0, k;
  } full[2];
  auto drain = [&](int h) -> int {
    HIPCHK(s.wait(h));
    auto& f = full[h];
    if (f.m > 0)
      runs(s.piece(h), out, n, f.q0, f.m, f.c0, f.k,
           [](const double* p, double* a, size_t count) { std::memcpy(a, p, count * sizeof(double)); });
    f.m = 0;
    return 0;
  };
  int last = 0;
  const int rc = Pieces(n, nc).each([&](int h, int q0, int m, int c0, int k) -> int {
    if (int rc = drain(h)) return rc;
    launch_rows_out(st_, m, k, map + q0, A ? A + c0 : nullptr, lda, B ? B + c0 : nullptr, ldb,
                    reinterpret_cast<double*>(s.piece(h)), m);
    HIPCHK(hipGetLastError());
    HIPCHK(s.mark(h, st_));
    full[h] = {q0, m, c0, k};
    last = h;
    return 0;
  });
  if (rc) return rc;
  if (int rc2 = drain(last ^ 1)) return rc2;
  return drain(last);
}

// The host's column-major n x nc array into rows map[0..n) (null: 0..n-1) of
// the row-major out, the other way through the same pieces.
int DeviceReducer::host_to_rows(int n, int nc, const int* map, const double* in, double* out, int ldo,
                                std::string& err) const {
  Stage& s = d_->stage;
  HIPCHK(s.open());
  return Pieces(n, nc).each([&](int h, int q0, int m, int c0, int k) -> int {
    HIPCHK(s.wait(h));
    runs(s.piece(h), const_cast<double*>(in), n, q0, m, c0, k,
         [](double* p, const double* a, size_t count) { std::memcpy(p, a, count * sizeof(double)); });
    launch_rows_in(st_, m, k, map ? map + q0 : nullptr, reinterpret_cast<const double*>(s.piece(h)), m,
                   out + c0 + (map ? 0 : (size_t)q0 * ldo), ldo);
    HIPCHK(hipGetLastError());
    HIPCHK(s.mark(h, st_));
    return 0;
  });
}

int DeviceReducer::get_B(double* B) const {
  std::string err;
  return rows_to_host(sym_.ndof1, sym_.ndof2, d_->p1.p, d_->X.p, sym_.ndof2, nullptr, 0, B, err);
}

int DeviceReducer::get_phi(double* P) const {
  std::string err;
  return rows_to_host(sym_.ndof1, res_.nev, d_->p1.p, d_->Phi.p, res_.nev, nullptr, 0, P, err);
}

int DeviceReducer::get_schur(std::vector<double>& S) {
  const Symbolic& y = sym_;
  const int n2 = y.ndof2;
  std::vector<double> f((size_t)n2 * n2);
  S.assign((size_t)n2 * n2, 0.0);
  if (n2 == 0) return 0;
  if (d_->mixed) {  // from the refined B (symmetric)
    S = d_->s22;
    return 0;
  }
  if (d2h(f.data(), d_->pool.p + y.foff[y.nsup - 1], sizeof(double) * f.size()) != hipSuccess)
    return -3;
  for (int j = 0; j < n2; j++)
    for (int i = 0; i < n2; i++) S[i + (size_t)j * n2] = i >= j ? f[i + (size_t)j * n2] : f[j + (size_t)i * n2];
  return 0;
}

int DeviceReducer::get_csr(std::vector<int>& rowptr, std::vector<int>& colind, std::vector<double>& K,
                           std::vector<double>& M) {
  const Symbolic& y = sym_;
  rowptr = y.rowptr;
  size_t nnz = y.rowptr[y.neq];
  colind.resize(nnz);
  K.resize(nnz);
  M.resize(nnz);
  if (d2h(colind.data(), d_->colind.p, sizeof(int) * nnz) != hipSuccess) return -3;
  if (d2h(K.data(), d_->Kv.p, sizeof(double) * nnz) != hipSuccess) return -3;
  if (d2h(M.data(), d_->Mv.p, sizeof(double) * nnz) != hipSuccess) return -3;
  return 0;
}

int DeviceReducer::get_element_matrices(std::vector<double>& Kp, std::vector<double>& Mp) {
  Kp.resize(sym_.elem_pool);
  Mp.resize(sym_.elem_pool);
  if (d2h(Kp.data(), d_->Kp.p, sizeof(double) * Kp.size()) != hipSuccess) return -3;
  if (d2h(Mp.data(), d_->Mp.p, sizeof(double) * Mp.size()) != hipSuccess) return -3;
  return 0;
}

// K_ii^-1 R into row-major x = d.sk_x (rows in elimination order), R as the
// caller's column-major n1 x nrhs, which has been read when the call returns.
int DeviceReducer::solve_rows(int nrhs, const double* R_eq, std::string& err) {
  Impl& d = *d_;
  const Symbolic& y = sym_;
  const int neq = y.neq, n1 = y.ndof1;
  SolvePlan* p = nullptr;
  if (get_plan(y, d, nrhs, p, err)) return -3;
  if (ensure_work(d, std::max(nrhs, std::max(y.ndof2, opt_.lanczos_block)), err)) return -3;
  const size_t n = (size_t)neq * nrhs;
  HIPCHK(d.sk_r.alloc(n));
  HIPCHK(d.sk_t.alloc(n));
  HIPCHK(d.sk_x.alloc(n));
  if (int rc = host_to_rows(n1, nrhs, d.p1.p, R_eq, d.sk_r.p, nrhs, err)) return rc;
  launch_fill(st_, d.sk_r.p + (size_t)n1 * nrhs, (int64_t)(neq - n1) * nrhs, 0.0);
  return solve_int(st_, d, y, opt_, *p, d.sk_r.p, d.sk_t.p, d.sk_x.p, nullptr, err);
}

int DeviceReducer::solve_kii(int nrhs, const double* R_eq, double* X_eq, std::string& err) {
  StreamScope scope(st_);
  Impl& d = *d_;
  const int n1 = sym_.ndof1;
  if (n1 == 0) return 0;
  if (int rc = solve_rows(nrhs, R_eq, err)) return rc;
  return rows_to_host(n1, nrhs, d.p1.p, d.sk_x.p, nrhs, nullptr, 0, X_eq, err);
}

int DeviceReducer::gravity_internal(double* gi, std::string& err) {
  StreamScope scope(st_);
  Impl& d = *d_;
  const Symbolic& y = sym_;
  if (opt_.no_mass) { err = "gravity forces need the mass matrix"; return -1; }
  DBuf<double>& g = d.gi_g;
  HIPCHK(g.alloc((size_t)y.neq * 3));
  mass_mm(st_, y.neq, d, 3, d.grav.p, 3, g.p, 3);
  return rows_to_host(y.ndof1, 3, d.p1.p, g.p, 3, nullptr, 0, gi, err);
}

int DeviceReducer::reduce_loads(int nrhs, const double* F_eq, std::vector<double>& out, std::string& err) {
  StreamScope scope(st_);
  Impl& d = *d_;
  const Symbolic& y = sym_;
  const int neq = y.neq, n2 = y.ndof2, ngen = res_.ngen, nev = res_.nev, nd = res_.ndim;
  out.assign((size_t)nd * std::max(nrhs, 0), 0.0);
  if (nrhs <= 0) return 0;
  if (out.empty()) return 0;
  // the products of reduce_loads_noalloc on buffers of the handle; the load
  // vectors cross the bus in the caller's order, the result once
  const size_t nF = (size_t)neq * nrhs, maxa = (size_t)std::max(n2, ngen), nout = out.size() * sizeof(double);
  HIPCHK(d.rl_f.alloc(nF));
  HIPCHK(d.part.alloc((size_t)xty_chunks(neq) * maxa * nrhs));
  HIPCHK(d.acc.alloc((size_t)(n2 + ngen + nd) * nrhs));
  double *const f = d.rl_f.p, *const r2 = d.acc.p, *const r1 = r2 + (size_t)n2 * nrhs;
  if (int rc = host_to_rows(neq, nrhs, d.e2p.p, F_eq, f, nrhs, err)) return rc;
  // rhs2 = f_e + B^T f_i = [B; I]^T f, rhs1 = Phi^T f_i
  if (n2 > 0) launch_xty(st_, neq, n2, nrhs, d.X.p, n2, f, nrhs, d.part.p, r2);
  if (ngen > 0) launch_xty(st_, neq, ngen, nrhs, d.Phi.p, nev, f, nrhs, d.part.p, r1);
  // written straight into pinned memory where it fits
  const bool small = nout <= Stage::PIECE;
  if (small) HIPCHK(d.stage.wait(0));
  double* const red = small ? reinterpret_cast<double*>(d.stage.piece(0)) : r1 + (size_t)ngen * nrhs;
  launch_scatter_reduced(st_, nd, n2, ngen, nrhs, d.pos2.p, r2, r1, red);
  HIPCHK(hipGetLastError());
  if (small) {
    HIPCHK(hipStreamSynchronize(st_));
    std::memcpy(out.data(), red, nout);
  } else {
    HIPCHK(d2h(out.data(), red, nout));
  }
  return 0;
}

// reduce_loads on device buffers, with every work buffer in the library's
// static scratch array: no device allocation.  F (neq x nrhs) and Fred
// (ndim x nrhs) are column-major device arrays.
int DeviceReducer::reduce_loads_noalloc(int nrhs, const double* F, double* Fred, std::string& err) {
  StreamScope scope(st_);
  Impl& d = *d_;
  const Symbolic& y = sym_;
  const int neq = y.neq, n2 = y.ndof2, ngen = res_.ngen, nev = res_.nev, nd = res_.ndim;
  double* scr = nullptr;
  size_t cap = 0;
  if (int rc = noalloc_scratch(&scr, &cap, err)) return rc;
  const size_t nF = (size_t)neq * nrhs, maxa = (size_t)std::max(n2, ngen);
  const size_t npart = (size_t)xty_chunks(neq) * maxa * nrhs;
  const size_t need = 8 * (nF + npart + (size_t)(n2 + ngen) * nrhs);
  if (need > cap) {
    err = "reduced loads without allocation: " + std::to_string(nrhs) + " load cases need " + std::to_string(need) +
          " bytes of scratch, more than the " + std::to_string(cap) + " available";
    return -1;
  }
  double* Fp = scr;
  double* part = Fp + nF;
  double* r2 = part + npart;
  double* r1 = r2 + (size_t)n2 * nrhs;
  launch_rows_in(st_, neq, nrhs, d.e2p.p, F, neq, Fp, nrhs);
  if (n2 > 0) launch_xty(st_, neq, n2, nrhs, d.X.p, n2, Fp, nrhs, part, r2);
  if (ngen > 0) launch_xty(st_, neq, ngen, nrhs, d.Phi.p, nev, Fp, nrhs, part, r1);
  launch_scatter_reduced(st_, nd, n2, ngen, nrhs, d.pos2.p, r2, r1, Fred);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(st_));
  return 0;
}

int DeviceReducer::recover(int nrhs, const double* Ub, const double* Fi, double* Ui, std::string& err) {
  StreamScope scope(st_);
  Impl& d = *d_;
  const Symbolic& y = sym_;
  const int neq = y.neq, n1 = y.ndof1, n2 = y.ndof2;
  if (nrhs <= 0) return 0;
  const bool bound = n2 > 0 && Ub;
  if (n1 == 0) return 0;
  if (!bound && !Fi) {
    std::fill(Ui, Ui + (size_t)n1 * nrhs, 0.0);
    return 0;
  }
  // x = K_ii^-1 F_i first, then per column chunk Y = [B; I] U_b and the sum of
  // both in the caller's order
  if (Fi)
    if (int rc = solve_rows(nrhs, Fi, err)) return rc;
  const int cj = bound ? std::min(nrhs, 64) : nrhs;
  if (bound) {
    HIPCHK(d.rc_s.alloc((size_t)n2 * cj));
    HIPCHK(d.rc_y.alloc((size_t)neq * cj));
  }
  for (int j0 = 0; j0 < nrhs; j0 += cj) {
    const int nj = std::min(cj, nrhs - j0);
    if (bound) {
      if (int rc = host_to_rows(n2, nj, nullptr, Ub + (size_t)j0 * n2, d.rc_s.p, nj, err)) return rc;
      launch_gemm_small(st_, neq, n2, nj, d.X.p, n2, d.rc_s.p, d.rc_y.p, nj, 0.0, 1.0);
    }
    if (int rc = rows_to_host(n1, nj, d.p1.p, bound ? d.rc_y.p : nullptr, nj, Fi ? d.sk_x.p + j0 : nullptr, nrhs,
                              Ui + (size_t)j0 * n1, err))
      return rc;
  }
  return 0;
}

int DeviceReducer::autotune(int& panel, int& split, std::string& err) {
  Impl& d = *d_;
  if (!uploaded_ && upload(err)) return -3;
  auto set_panel = [&](int P) -> int {
    std::vector<FTask> ft;
    std::vector<int> xr;
    d.fops.clear();
    build_factor_schedule(sym_, d.lay, ft, d.fops, xr, upd_flops_, P, opt_.factor_lookahead);
    HIPCHK(ensure_side(d));
    HIPCHK(d.ftasks.upload(ft));
    HIPCHK(d.xrange.upload(xr));
    upd_launches_ = 0;
    for (auto& op : d.fops)
      if (op.kind == UPDATE || op.kind == UPDATE_SIDE) upd_launches_++;
    d.g_factor.reset();
    opt_.factor_panel = P;
    return 0;
  };
  auto set_split = [&](int KS) {
    d.solve_split = KS;
    opt_.solve_split = KS;
    d.plans.clear();
    };
  // warm-up (allocations, first captures), then one timed reduction per candidate
  if (int rc = reduce(err)) return rc;
  double best = INFINITY;
  int bestP = 256;
  for (int P : {64, 128, 192, 256}) {
    if (set_panel(P)) return -3;
    if (int rc = reduce(err)) return rc;
    if (int rc = reduce(err)) return rc;  // the second run replays the captured factor graph
    if (times_.factor < best) { best = times_.factor; bestP = P; }
  }
  if (set_panel(bestP)) return -3;
  best = INFINITY;
  int bestK = d.solve_split;
  for (int KS : {64, 128, 256, 512}) {
    set_split(KS);
    if (int rc = reduce(err)) return rc;
    if (int rc = reduce(err)) return rc;
    const double t = times_.bsolve + times_.modes;
    if (t < best) { best = t; bestK = KS; }
  }
  set_split(bestK);
  panel = bestP;
  split = bestK;
  return 0;
}

// The buffers of upload(), reduce() and, for nlc load cases, reduce_loads() and
// recover(), in that order; task lists and index arrays of a few bytes per
// front row or node are taken as a whole.
size_t DeviceReducer::footprint_bytes(int nlc) const {
  const Symbolic& y = sym_;
  const size_t neq = y.neq, n1 = y.ndof1, n2 = y.ndof2, nel = part_.nel, nnod = part_.nnod;
  const size_t nnz = y.rowptr.empty() ? 0 : (size_t)y.rowptr.back();
  const size_t ngen = opt_.ngen, lb = opt_.lanczos_block, ncases = std::max(nlc, 0);
  const size_t nev = ngen > 0 ? std::max(opt_.neval, opt_.ngen) : 0;
  int bs = 0, cap = 0;
  if (nev > 0 && n1 > 0) lanczos_sizes(y.ndof1, (int)nev, opt_, bs, cap);
  const size_t nb = bs, mcap = cap, chunks = xty_chunks(y.neq), f8 = sizeof(double), fb = opt_.mixed ? 4 : 8;
  const SolveLayout lay = solve_layout(y, opt_);
  size_t wrows = 0, tasks = 0;
  for (int s = 0; s < y.nsup; s++) {
    const size_t T = (y.nrow[s] + 63) / 64, C = (y.ncol[s] + 63) / 64;
    wrows += y.nrow[s];
    tasks += y.nrow[s] / 8 + C * (2 * T + C);  // cleared and gathered columns, inverse and panel tiles
    for (size_t c = 0; c < C; c++) tasks += 5 * (T - c) + (c % 4 == 0 ? (T - c) * (T - c) / 2 : 0);  // factor
  }
  // part, structure, schedules
  size_t b = nnod * 48 + nel * (f8 * NPROP + 32) + 4 * part_.enodes.size() + 40 * neq + 8 * y.nbl.size();
  b += 8 * sam_.msc.size() + 20 * sam_.ceq_dof.size() + 4 * sam_.ceq_ptr.size();
  b += 60 * (size_t)y.nsup + 4 * (y.rows.size() + 2 * y.rel.size()) + 12 * wrows;
  b += (y.has_rigid ? 12 : 4) * (size_t)y.ncontrib + nnz * (4 + 4 + 8 + 4);
  b += sizeof(FTask) * tasks + 12 * (wrows / 8 + y.rel.size() / 16) + 3 * 24 * wrows;
  // factor, matrices
  b += fb * ((size_t)y.fpool + (size_t)lay.ioff[y.nsup]) + f8 * inverse_workspace(y);
  b += f8 * (2 * (size_t)y.elem_pool + 2 * nnz + 2 * n1);
  // solves: the widest of B, the Lanczos block, the gravity displacements and the load cases
  const size_t wide = std::max({n2, ncases > 0 ? std::max(ncases, lb) : (size_t)0, nev > 0 ? std::max(nb, n2) : (size_t)0,
                                opt_.want_vgi ? std::max<size_t>(3, lb) : (size_t)0});
  b += f8 * wrows * wide * (lay.unfused ? 2 : 1);
  b += f8 * neq * 3 * n2;
  if (nev > 0) {
    b += f8 * neq * (2 * mcap + nb + std::max(nb, opt_.want_vgi ? std::max<size_t>(3, lb) : 0) + std::max(nb, std::max(ngen, lb)) + nev);
    b += f8 * (mcap * std::max(nb, nev) + mcap * mcap + mcap * nb + nev * (1 + 3 * MODE_SIGN_GROUPS));
  }
  if (opt_.want_vgi) b += f8 * neq * 2 * std::max<size_t>(3, lb);
  if (!opt_.no_mass) b += f8 * neq * std::max<size_t>(3, std::max(lb, nev));
  // products: the partial sums of the largest
  const size_t ab = std::max(std::max<size_t>(n2, 3), std::max<size_t>(nev, 1));
  b += f8 * chunks * std::max({ab * ab, mcap * std::max(nb, nev), std::max(n2, ngen) * ncases});
  b += f8 * (3 * (n2 + ngen + 6) * (n2 + ngen + 6) + (2 * (n2 + ngen) + 6) * ncases);
  if (opt_.mixed) b += f8 * neq * (1 + 5 * wide);
  if (ncases > 0) b += f8 * (neq * (4 * ncases + std::min<size_t>(ncases, 64)) + n2 * std::min<size_t>(ncases, 64));
  return b;
}

}  // namespace fgpu
