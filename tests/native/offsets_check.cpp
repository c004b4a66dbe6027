// The level-piece kernels' base-state accesses on grids whose levels span more than 2^32 bytes, on the host: an x-z slice
// of 2^29 elements and more per field (its full base state a sparse mapping, one value written per place read), a 3-D
// domain's rows and a horizontally uniform profile, against BField's own index.
#include <sys/mman.h>

#include <cstdio>
#include <vector>

#include "../../cppwrf_amd/csrc/dev_common.hpp"

using namespace mi_dev;

static int bad = 0;

// nx x nz of a slice (rows = 1), or ny rows with the halo of 3
static void full_field(int nx, int ny, int nz) {
  const int64_t sk = (int64_t(kLpad) + nx + 1 + kHalo + 31) / 32 * 32, block = sk * (nz + 1);
  const int rows = ny == 1 ? 1 : ny + 1 + 2 * kHalo, hy = ny == 1 ? 0 : kHalo;
  const size_t bytes = size_t(block) * size_t(rows) * sizeof(double);
  void* m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (m == MAP_FAILED) {
    std::printf("%dx%dx%d: no address space for %zu bytes\n", nx, ny, nz, bytes);
    ++bad;
    return;
  }
  const idx_t sj = ny == 1 ? 0 : idx_t(block);
  double* p = static_cast<double*>(m) + kLpad + int64_t(hy) * sj;
  const BField b{p, 1, sj, idx_t(sk)};
  const int is[] = {0, 1, nx / 2, nx - 1, nx}, js[] = {0, ny / 2, ny - 1}, ks[] = {0, 1, nz / 2, nz - 1};
  double next = 1;
  for (int j : js)
    for (int k : ks)
      for (int i : is) p[int64_t(i) + int64_t(j) * sj + int64_t(k) * sk] = next++;
  for (int j : js)
    for (int k : ks)
      for (int i : is) {
        // the arguments of advance_uv and of the tendencies of u and v: the row's start, the lane's offset in it
        const double got = BaseLevels(b, j * sj - kLpad, unsigned(kLpad + i))(k), want = p[int64_t(i) + int64_t(j) * sj + int64_t(k) * sk];
        if (got != want && bad++ < 8)
          std::printf("%dx%dx%d: base state at (%d, %d, %d): %g, not %g\n", nx, ny, nz, i, j, k, got, want);
      }
  munmap(m, bytes);
}

int main() {
  full_field(97, 75, 35);
  full_field(300, 1, 10);
  full_field(1 << 23, 1, 62);  // a little below 2^29 elements
  full_field(1 << 23, 1, 64);  // above
  full_field(8000000, 1, 255);  // 2^31 elements less 4 %
  std::vector<double> prof(64);
  for (int k = 0; k < 64; ++k) prof[size_t(k)] = 1000.0 + k;
  const BField b{prof.data(), 0, 0, 1};
  for (int k = 0; k < 64; ++k)
    if (BaseLevels(b, 12345, 678u)(k) != prof[size_t(k)]) ++bad;
  std::printf("%d wrong\n", bad);
  return bad ? 1 : 0;
}
