// Plans of several problems, built on the host with the library's own planner
// and printed one launch a line:
//   plan_probe f64|f32 [problem ...]
// problem: m,k,n[,algorithm,steps[,depth-first levels]]; the algorithm blocks:MxKxN is
// the classical product of an M x K by K x N split (a plan only: it has no kernels)
//   gemm cfg any full products tiles max_k_of_products
//   thin products tiles
//   stage kind nodes k_updates peeling_products
//   peel kind M N K c_offset c_ld (each product of the launch above)
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "plan.hpp"

using namespace fmplan;

extern const FmAlgDesc* fm_find_alg(const char* name);

namespace {
double one(int, double) { return 1.0; }

FmAlgDesc* classical(int m, int k, int n) {
  FmAlgDesc* d = new FmAlgDesc();
  memset(d, 0, sizeof(*d));
  d->name = "blocks";
  d->m = m;
  d->k = k;
  d->n = n;
  d->R = m * k * n;
  int *kind = new int[(size_t)d->R](), *a = new int[(size_t)d->R], *b = new int[(size_t)d->R];
  for (int r = 0, i = 0; i < m; ++i)
    for (int j = 0; j < n; ++j)
      for (int q = 0; q < k; ++q, ++r) {
        a[r] = i * k + q;
        b[r] = q * n + j;
      }
  d->a_kind = d->b_kind = kind;
  d->a_index = a;
  d->b_index = b;
  d->a_coef = d->b_coef = one;
  return d;
}
}  // namespace

int main(int argc, char** argv) {
  const fm_dtype dt = strcmp(argv[1], "f64") == 0 ? FM_F64 : FM_F32;
  Plan P;
  P.dtype = dt;
  std::vector<SubPlan> subs((size_t)(argc - 2));
  int64_t ws = 0;
  for (int i = 0; i < argc - 2; ++i) {
    std::vector<std::string> f;
    for (char* t = strtok(argv[i + 2], ","); t; t = strtok(nullptr, ",")) f.push_back(t);
    Problem p;
    p.m = p.lda = p.ldc = atoll(f[0].c_str());
    p.k = p.ldb = atoll(f[1].c_str());
    p.n = atoll(f[2].c_str());
    p.role_a = 4 + 3 * i;
    p.role_b = 5 + 3 * i;
    p.role_c = 6 + 3 * i;
    if (f.size() > 4) {
      int bm, bk, bn;
      if (sscanf(f[3].c_str(), "blocks:%dx%dx%d", &bm, &bk, &bn) == 3)
        p.alg = classical(bm, bk, bn);
      else
        p.alg = fm_find_alg(f[3].c_str());
      p.steps = atoi(f[4].c_str());
      if (!p.alg) return 2;
    }
    if (f.size() > 5) p.dfs = atoi(f[5].c_str());
    if (build_subplan(dt, p, ws, subs[(size_t)i]) != FM_OK) {
      fprintf(stderr, "%s\n", last_error().c_str());
      return 1;
    }
    ws += subs[(size_t)i].ws_elems;
  }
  if (assemble(P, subs, ws) != FM_OK) {
    fprintf(stderr, "%s\n", last_error().c_str());
    return 1;
  }
  for (const Launch& L : P.launches) {
    if (L.kind == LK_GEMM) {
      int k = 0;
      for (const FmGemmDesc& d : L.gdescs) k = std::max(k, d.K);
      printf("gemm %d %d %d %d %d %d\n", L.cfg, L.gm.any, L.gm.full, L.gm.ndesc, L.gm.total_tiles, k);
    } else if (L.kind == LK_THIN) {
      printf("thin %d %d\n", L.th.ndesc, L.th.total_tiles);
    } else {
      printf("stage %d %d %d %d\n", (int)L.kind, L.st.nodes, L.nupd, (int)L.tdescs.size());
    }
    for (const FmThinDesc& d : L.tdescs)
      printf("peel %d %d %d %d %lld %lld\n", (int)d.kind, d.M, d.N, d.K, (long long)d.c.off, (long long)d.c.ld);
  }
  return 0;
}
