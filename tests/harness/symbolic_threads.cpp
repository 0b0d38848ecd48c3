// Ordering and front lists of the part on stdin (node count, element count,
// leaf size; per node x y z status; per element type and 1-based nodes) with
// 1, 2, 4, 7 and 8 threads: prints the number of fronts, the most children of
// one, and the lists that differ from those of one thread ("same" if none).
#include <cstdio>
#include <string>
#include "../../fedem-solvers_amd/csrc/fgpu.hpp"

int main() {
  using namespace fgpu;
  Part p;
  SymbolicOptions o;
  if (std::scanf("%d %d %d", &p.nnod, &p.nel, &o.leaf_nodes) != 3) return 1;
  p.xyz.resize(3 * p.nnod);
  p.status.resize(p.nnod);
  for (int i = 0; i < p.nnod; i++)
    if (std::scanf("%lf %lf %lf %d", &p.xyz[3 * i], &p.xyz[3 * i + 1], &p.xyz[3 * i + 2], &p.status[i]) != 4) return 1;
  p.eptr.assign(1, 0);
  for (int e = 0; e < p.nel; e++) {
    int t = 0, n = 0;
    if (std::scanf("%d", &t) != 1) return 1;
    p.etype.push_back(t);
    for (int k = 0; k < elem_nodes(t); k++) {
      if (std::scanf("%d", &n) != 1) return 1;
      p.enodes.push_back(n - 1);
    }
    p.eptr.push_back((int)p.enodes.size());
  }
  p.eprop.assign((size_t)NPROP * p.nel, 1.0);
  Sam sam;
  std::string err;
  if (build_sam(p, sam, err)) return 2;
  Symbolic a;
  o.threads = 1;
  if (build_symbolic(p, sam, o, a, err)) return 3;
  int most = 0;
  for (int s = 0; s < a.nsup; s++)
    if (a.chptr[s + 1] - a.chptr[s] > most) most = a.chptr[s + 1] - a.chptr[s];
  std::printf("%d %d", a.nsup, most);
  std::string bad;
  for (int threads : {2, 4, 7, 8}) {
    Symbolic b;
    o.threads = threads;
    if (build_symbolic(p, sam, o, b, err)) return 4;
#define SAME(x) \
  if (!(a.x == b.x)) bad += " " #x;
    SAME(eq_to_perm) SAME(perm_to_eq) SAME(elem_off) SAME(elem_pool) SAME(rowptr) SAME(nfirst) SAME(neqd) SAME(nrow0)
    SAME(nbptr) SAME(nbl) SAME(rnode) SAME(colsn) SAME(drank) SAME(ncontrib) SAME(nsup) SAME(col0) SAME(ncol)
    SAME(nrow) SAME(parent) SAME(level) SAME(rptr) SAME(rows) SAME(foff) SAME(fpool) SAME(chptr) SAME(chlist)
    SAME(relptr) SAME(rel) SAME(nlevels) SAME(lvptr) SAME(lvsup) SAME(factor_flops) SAME(nnzL) SAME(maxfront)
  }
  std::printf(" %s\n", bad.empty() ? "same" : bad.c_str());
  return 0;
}
