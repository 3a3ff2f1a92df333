// Host program for tests/test_gemm_plans.py: prints the plan (tile, splits) that
// gemm_plan gives each contraction read from standard input.  Only the plan is
// computed: pointers are aligned placeholders and nothing is launched.
#include <cstdio>

#include "di_gemm.h"

int main() {
  // elem (0 fp32, 1 fp16), b_mode, CUs, batch, M, N, K, act, then for a conv its
  // input channels (0: dense), size, kernel, stride and upsampling, and whether
  // row statistics are wanted
  unsigned elem, b_mode, cus, batch, M, N, K, act, cin, h, w, ks, stride, up, rstats;
  while (scanf("%u %u %u %u %u %u %u %u %u %u %u %u %u %u %u", &elem, &b_mode, &cus, &batch, &M, &N,
               &K, &act, &cin, &h, &w, &ks, &stride, &up, &rstats) == 15) {
    di::GemmArgs g;
    if (rstats) g.rstats = (float*)4096;
    const uint64_t es = elem ? 2 : 4;
    g.a = g.b = g.c = (void*)4096;
    g.batch = batch;
    g.M = M;
    g.N = N;
    g.K = K;
    g.act = (int)act;
    g.lda = g.ldb = K;
    if (b_mode == di::B_KN) g.ldb = N;
    g.ldc = act == di::ACT_GEGLU ? N / 2 : N;
    g.sc = (uint64_t)M * N;
    g.c_f32 = !elem;
    g.a_vec_ok = K % (16 / es) == 0;
    g.b_vec_ok = g.ldb % (16 / es) == 0;
    g.a_bytes = di::gemm_extent((uint64_t)M * K * es);
    if (cin) {
      g.Cin = cin;
      g.H = h;
      g.W = w;
      g.ks = ks;
      g.stride = stride;
      g.pad = ks / 2;
      g.up = up;
      g.Ho = (h * up + 2 * g.pad - ks) / stride + 1;
      g.Wo = (w * up + 2 * g.pad - ks) / stride + 1;
      g.lda = cin;
      g.c_nchw = !elem;
      g.a_bytes = di::gemm_extent((uint64_t)(M / (g.Ho * g.Wo)) * h * w * cin * es);
    }
    g.b_bytes = di::gemm_extent((uint64_t)N * K * es);
    const di::GemmPlan p = di::gemm_plan(g, elem ? 1 : 0, (int)cus, (int)b_mode);
    printf("%d %u\n", p.tile, p.splits);
  }
  return 0;
}
