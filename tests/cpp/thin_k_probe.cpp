// One peeling update C = alpha A B + beta C through the library's thin kernels, on
// small whole numbers, against the same product on the host:
//   thin_k_probe f64|f32 M N K beta
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "gemm_thin.hpp"

template <typename T>
static int run(int f64, int M, int N, int K, double beta) {
  const int64_t lda = M + 3, ldb = K + 1, ldc = M + 2;
  std::vector<T> A(lda * K), B(ldb * N), C(ldc * N), want(C.size()), got(C.size());
  unsigned s = 12345;
  auto fill = [&](std::vector<T>& v) {
    for (T& x : v) {
      s = s * 1664525u + 1013904223u;
      x = (T)((int)(s >> 24) % 17 - 8);
    }
  };
  fill(A);
  fill(B);
  fill(C);
  want = C;
  for (int j = 0; j < N; ++j)
    for (int i = 0; i < M; ++i) {
      double t = 0;
      for (int k = 0; k < K; ++k) t += (double)A[i + k * lda] * (double)B[k + j * ldb];
      want[i + j * ldc] = (T)(2.0 * t + beta * (double)C[i + j * ldc]);
    }
  FmThinDesc d;
  memset(&d, 0, sizeof(d));
  d.a.ld = lda;
  d.b.ld = ldb;
  d.c.ld = ldc;
  d.a.role = 0;
  d.b.role = 1;
  d.c.role = 2;
  d.M = M;
  d.N = N;
  d.K = K;
  d.kind = FM_THIN_K;
  d.alpha = 2.0;
  d.beta = beta;
  int bm, bn;
  fm_thin_tile(f64, FM_THIN_K, K, &bm, &bn);
  d.tiles_m = (M + bm - 1) / bm;
  FmThinArgs a;
  memset(&a, 0, sizeof(a));
  a.ndesc = 1;
  a.uniform = 1;
  a.total_tiles = a.per[0] = a.t0[1] = a.t0[2] = d.tiles_m * ((N + bn - 1) / bn);
  a.per[1] = a.per[2] = a.d0[1] = a.d0[2] = 1;
  void* p[4];
  const void* src[4] = {A.data(), B.data(), C.data(), &d};
  const size_t bytes[4] = {A.size() * sizeof(T), B.size() * sizeof(T), C.size() * sizeof(T), sizeof(d)};
  for (int i = 0; i < 4; ++i) {
    if (hipMalloc(&p[i], bytes[i]) != hipSuccess) return 2;
    if (hipMemcpy(p[i], src[i], bytes[i], hipMemcpyHostToDevice) != hipSuccess) return 2;
  }
  for (int i = 0; i < 3; ++i) a.bases.p[i] = p[i];
  a.descs = (const FmThinDesc*)p[3];
  if (fm_thin_launch(f64, a, nullptr) != hipSuccess) return 3;
  if (hipMemcpy(got.data(), p[2], bytes[2], hipMemcpyDeviceToHost) != hipSuccess) return 3;
  for (void* q : p) (void)hipFree(q);
  return memcmp(got.data(), want.data(), bytes[2]) == 0 ? 0 : 1;
}

int main(int argc, char** argv) {
  if (argc < 6) return 4;
  const int f64 = strcmp(argv[1], "f64") == 0, M = atoi(argv[2]), N = atoi(argv[3]), K = atoi(argv[4]);
  const int r = f64 ? run<double>(f64, M, N, K, atof(argv[5])) : run<float>(f64, M, N, K, atof(argv[5]));
  printf("%d\n", r);
  return r;
}
