// The library's choice of the substep kernel's form, for a domain alone and for a batch, on grids whose row block is
// below, at and above 2^29 elements: the form with several levels per thread reaches it with 32-bit byte offsets.  Built
// for each arithmetic (MI_REAL, MI_NS) and linked with the library; nothing is launched.
#include <cstdio>

#include "../../cppwrf_amd/csrc/kernels_fp64.hpp"

using namespace MI_NS;

static Args grid(int64_t sk, int nz, bool slice) {
  Args a{};
  a.g.nz = nz;
  a.g.sk = mi_dev::idx_t(sk);
  a.g.sj = slice ? 0 : mi_dev::idx_t(sk * (nz + 1));
  a.g.ny = slice ? 1 : 100;
  a.g.two_d = slice;
  return a;
}

int main() {
  int bad = 0;
  const bool f32 = sizeof(real) == 4;
  auto expect = [&](const char* what, int got, int want) {
    if (got != want) {
      std::printf("%s: %d, not %d\n", what, got, want);
      ++bad;
    }
  };
  const Args small = grid(352, 44, false), below = grid((1 << 23) - 32, 63, true), at = grid(1 << 23, 63, true),
             above = grid((1 << 23) + 32, 62, true), tall = grid(1 << 22, 127, true), taller = grid(1 << 22, 128, true);
  for (const Args* a : {&small, &below}) {
    expect("a small row block", acoustic_cfg(*a, kColLevels), kColLevels);
    const Args* one[] = {a};
    expect("a batch of small row blocks", batch_levels(one, 1), f32);
  }
  expect("63 levels", acoustic_cfg(at, kColLevels), 4);
  expect("62 levels", acoustic_cfg(above, kColLevels), kColLevels);  // 63 rows of it: less than 2^29
  expect("127 levels", acoustic_cfg(tall, kColLevels), 5);
  expect("128 levels", acoustic_cfg(taller, kColLevels), 6);
  for (int cfg = 0; cfg < kNumColCfgs; ++cfg) expect("a shape of one level per thread", acoustic_cfg(at, cfg), cfg);
  const Args* mixed[] = {&small, &below, &at};
  expect("two small members", batch_levels(mixed, 2), f32);
  expect("a large member among small ones", batch_levels(mixed, 3), 0);
  std::printf("%d wrong\n", bad);
  return bad ? 1 : 0;
}
