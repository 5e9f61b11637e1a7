// Checks the pieces of stage_plan.h: every part once and in order, whatever the
// sizes, and never more pinned memory than the ring has.
#include <stdio.h>
#include <stdint.h>
#include "../../dvc_amd/csrc/stage_plan.h"

using namespace dvc;

static int failures = 0;
static void expect(bool ok, const char *what, int n, int kind) {
  if (ok) return;
  printf("%s: %d parts, sizes %d\n", what, n, kind);
  failures++;
}

int main() {
  const size_t cif = 9u * 352 * 288, qcif = 9u * 176 * 144;
  uint64_t seed = 1;
  for (int n : {1, 2, 3, 4, 5, 7, 8, 9, 31, 32, 33, 64, 100, 1000, 5000})
    for (int kind = 0; kind < 5; kind++) {
      std::vector<size_t> at{512};
      for (int i = 0; i < n; i++) {
        seed = seed * 6364136223846793005ull + 1442695040888963407ull;
        const bool big = kind == 0 || (kind == 2 && i % 2) || (kind == 3 && i < n / 2) || (kind == 4 && (seed >> 40) % 3);
        const size_t whole = big ? cif : qcif;
        at.push_back(at.back() + (kind == 4 ? whole / 9 * ((seed >> 50) % 9 + 1) : whole));
      }
      const int want = std::min(8, (n + 3) / 4);
      const std::vector<int> cut = stage_pieces(at, want);
      expect(cut.front() == 0 && cut.back() == n, "ends", n, kind);
      for (size_t k = 0; k + 1 < cut.size(); k++) {
        expect(cut[k] < cut[k + 1], "empty piece", n, kind);
        expect(at[cut[k + 1]] - at[cut[k]] <= kStageSlot, "piece larger than a slot", n, kind);
      }
      expect(stage_slot_bytes(at, cut) <= kStageSlot, "slot", n, kind);
      // no more pieces than asked for while they fit, and not many more than fit
      const size_t total = at[n] - at[0];
      expect((int)cut.size() - 1 <= std::max<int>(want, (int)(total / (kStageSlot - cif)) + 1), "pieces", n, kind);
    }
  // 64 CIF pairs: eight pieces of eight
  std::vector<size_t> at{0};
  for (int i = 0; i < 64; i++) at.push_back(at.back() + cif);
  expect(stage_pieces(at, 8) == std::vector<int>({0, 8, 16, 24, 32, 40, 48, 56, 64}), "eights", 64, 0);
  expect(kStageSlots * kStageSlot <= (64u << 20), "ring", 0, 0);
  expect(si_result_bytes(100, false, false) == 100 && si_result_bytes(100, true, false) == 500 &&
             si_result_bytes(100, false, true) == 500 && si_result_bytes(100, true, true) == 900,
         "result bytes", 0, 0);
  puts(failures ? "FAILED" : "ok");
  return failures != 0;
}
