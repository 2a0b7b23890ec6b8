// Host-side check of the fp32 prefill's dispatch order (dealt_item in
// prefill_f32.hip), compiled from the kernel source and run on the CPU (no GPU
// call). Over random run lengths and grids: the order is a permutation of the
// grid, consecutive items of a run share an XCD, and a chunk's tiles at the same
// place of every turn reach at least half of the XCDs.
#include "prefill_f32.hip"

#include <cstdio>
#include <random>
#include <vector>

// The file's host launcher references this; nothing here launches.
namespace clv {
hipError_t launch_prefill_valu(const PrefillParams &, DType, hipStream_t) {
  return hipErrorInvalidValue;
}
}  // namespace clv

int main() {
  std::mt19937_64 rng(11);
  long cases = 0, bad = 0;
  for (int it = 0; it < 20000; ++it) {
    const int run = it % 3 == 0 ? 1 + (int)(rng() % 500) : 1 + (int)(rng() % 8);
    const int turns = 1 + (int)(rng() % 40);
    const int grid = 8 * run * turns;
    std::vector<int> xcd(grid, -1);
    bool ok = true;
    for (int b = 0; b < grid && ok; ++b) {
      const int l = clv::dealt_item(b, run);
      if (l < 0 || l >= grid || xcd[l] >= 0) ok = false;
      else xcd[l] = b % 8;
    }
    for (int l = 0; l + 1 < grid && ok; ++l)
      if (l % run != run - 1 && xcd[l] != xcd[l + 1]) ok = false;
    // Every step-th run (a chunk's tiles span whole turns or fractions of them).
    for (int step = 1; step <= 64 && ok; step *= 2) {
      std::vector<int> used(8, 0);
      int n = 0, kinds = 0;
      for (int u = 0; u < 8 * turns; u += step, ++n) kinds += used[xcd[u * run]]++ == 0;
      if (n >= 32 && kinds < 4) ok = false;
    }
    ++cases;
    if (!ok) {
      if (bad < 5) printf("bad: run %d turns %d\n", run, turns);
      ++bad;
    }
  }
  // One run per XCD is the contiguous order.
  for (int b = 0; b < 800; ++b)
    if (clv::dealt_item(b, 100) != b % 8 * 100 + b / 8) ++bad;
  printf("cases %ld bad %ld\n", cases, bad);
  return bad != 0;
}
