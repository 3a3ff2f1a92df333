// Host program for tests/test_workspace.py: what partials_workspace does where the
// workspace cannot grow.  No HIP call is reached.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "di_gemm.h"
#include "di_internal.h"

int main() {
  di::Ctx c;
  int bad = 0;
  auto expect = [&](bool ok, const char* what) {
    if (!ok) printf("wrong: %s\n", what), bad = 1;
  };
  auto problem = [](uint32_t splits) {
    di::GemmArgs g;
    g.M = 512;
    g.N = 512;
    g.K = 4096;
    g.splits = splits;
    return g;
  };
  di::GemmArgs g = problem(1);
  c.hold_releases = true;
  expect(di::partials_workspace(&c, g) == DI_OK && !g.part, "one piece needs no workspace");
  // growth during a graph capture is an error, not a reason for another plan
  g = problem(4);
  expect(di::partials_workspace(&c, g) == DI_EINVAL && g.splits == 4, "capture");
  // no memory: one piece
  c.hold_releases = false;
  setenv("DI_WORKSPACE_LIMIT", "4194303", 1);  // 4 x 512 x 512 floats need 4194304
  expect(di::partials_workspace(&c, g) == DI_OK && g.splits == 1 && !g.part, "no memory");
  void* p = nullptr;
  expect(di::workspace(&c, 1ull << 40, &p) == DI_ENOMEM &&
             strstr(di::get_error(), "DI_WORKSPACE_LIMIT"), "limit");
  // what is there is used
  c.ws = &g;
  c.ws_bytes = 4194304;
  g = problem(4);
  expect(di::partials_workspace(&c, g) == DI_OK && g.splits == 4 && g.part == c.ws, "fits");
  puts(bad ? "FAILED" : "OK");
  return bad;
}
