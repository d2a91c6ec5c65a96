// Host check of the rules that choose a handle's kernels: the shell sums' path
// (rmt_path) on both field layouts, and the far field's expansion, which must
// not bring in FP64 tables in global memory where the direct sums' fields need
// none.  Prints one line per failure and the counts.
#include "harmonic_plan.hpp"

#include <cstdio>

namespace glst {
std::string tdesign_dir() { return ""; }
namespace dev {
template <typename T>
size_t harm_lds_sf(uint32_t, uint32_t) { return 0; }
template <typename T>
size_t harm_lds_lr(uint32_t, uint32_t, uint32_t) { return 0; }
template size_t harm_lds_sf<float>(uint32_t, uint32_t);
template size_t harm_lds_sf<double>(uint32_t, uint32_t);
template size_t harm_lds_lr<float>(uint32_t, uint32_t, uint32_t);
template size_t harm_lds_lr<double>(uint32_t, uint32_t, uint32_t);
}  // namespace dev
}  // namespace glst

int main() {
  using namespace glst;
  using dev::RmtPath;
  constexpr size_t kLds = 160 * 1024;
  int failures = 0;
  long checks = 0, refused = 0;
  const uint32_t dims[] = {3, 4, 8, 9, 12, 15, 16, 17, 20, 21, 24, 33, 38, 64};
  for (bool mixed : {true, false})
    for (int shape = 0; shape <= 5; ++shape)
      for (uint32_t nx : dims)
        for (uint32_t ny : dims)
          for (uint32_t nz : dims) {
            const dev::GridShape g{nx, ny, nz, nx * ny * nz, 9.0};
            const RmtPath a = dev::rmt_path(mixed, shape, g, kLds, false);
            const RmtPath b = dev::rmt_path(mixed, shape, g, kLds, true);
            const bool fits = dev::rmt_nodes_per_group(nx, ny, nz, kLds, 1) > 0;
            // each path where its kernel takes the grid
            bool good = true;
            for (bool nm : {false, true}) {
              const RmtPath p = nm ? b : a;
              if (p == RmtPath::kMfma)
                good = good && mixed && dev::rmt_mfma_nodes(g, kLds, nm) > 0;
              if (p == RmtPath::kWave)
                good = good && mixed && dev::rmt_wave_fits(g);
              if (p == RmtPath::kLds) good = good && fits && shape != 2;
              if (p == RmtPath::kGlobal) good = good && (!fits || shape == 2);
            }
            const bool takes = harm_shell_sums(mixed, shape, g, kLds);
            const bool worse = b == RmtPath::kGlobal && a != RmtPath::kGlobal;
            if (!good || takes == worse) {
              std::printf("FAIL mixed %d shape %d grid %u x %u x %u: paths %d "
                          "%d takes %d\n", mixed, shape, nx, ny, nz,
                          static_cast<int>(a), static_cast<int>(b), takes);
              ++failures;
            }
            ++checks;
            refused += !takes;
          }
  auto refuses = [&](uint32_t nx, uint32_t ny, uint32_t nz, bool want) {
    const dev::GridShape g{nx, ny, nz, nx * ny * nz, 9.0};
    if (harm_shell_sums(true, 4, g, kLds) == want) {
      std::printf("FAIL %u x %u x %u\n", nx, ny, nz);
      ++failures;
    }
  };
  refuses(16, 16, 40, true);
  refuses(16, 16, 33, true);
  refuses(16, 16, 24, false);
  refuses(15, 15, 15, false);
  refuses(21, 21, 21, false);  // global tables on either layout
  // thin and small grids, rows of cells and node runs
  auto path = [&](uint32_t nx, uint32_t ny, uint32_t nz, bool nm, RmtPath want) {
    const dev::GridShape g{nx, ny, nz, nx * ny * nz, 9.0};
    if (dev::rmt_path(true, 4, g, kLds, nm) != want) {
      std::printf("FAIL path of %u x %u x %u, nm %d\n", nx, ny, nz, nm);
      ++failures;
    }
  };
  path(12, 12, 3, true, RmtPath::kLds);
  path(12, 12, 3, false, RmtPath::kMfma);
  path(3, 12, 12, true, RmtPath::kLds);
  path(12, 12, 6, true, RmtPath::kLds);
  path(16, 16, 8, true, RmtPath::kMfma);
  path(15, 15, 15, true, RmtPath::kMfma);
  path(9, 9, 9, true, RmtPath::kLds);
  path(6, 6, 6, true, RmtPath::kWave);
  path(16, 16, 24, true, RmtPath::kLds);
  path(16, 16, 24, false, RmtPath::kMfma);
  // dilute systems keep the direct sums: (charges, cells, nodes, mixed, taken)
  auto worth = [&](uint32_t n, uint32_t ncell, uint32_t K, bool mixed,
                   bool want) {
    if (harm_worth(n, ncell, K, mixed) != want) {
      std::printf("FAIL %u charges in %u cells\n", n, ncell);
      ++failures;
    }
  };
  worth(288000, 3375, 27453, true, true);
  worth(288000, 3375, 27453, false, true);
  worth(39304, 3375, 14718, true, false);
  worth(39304, 3375, 14718, false, false);
  worth(8000, 3375, 27453, true, false);
  worth(32928, 6144, 17862, true, false);
  worth(2744, 512, 74032, true, true);   // small grid
  worth(2744, 512, 200000, false, false);
  worth(10648, 512, 74032, false, true);
  worth(3000, 64, 20000, true, false);   // few pairs
  std::printf("checks %ld refused %ld failures %d\n", checks, refused, failures);
  return failures ? 1 : 0;
}
