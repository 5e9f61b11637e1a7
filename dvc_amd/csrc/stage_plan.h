// stage_plan.h -- how the results of a batch travel through a bounded ring of
// pinned slots; no GPU needed, so host tests compile it by itself.
#pragma once
#include <stddef.h>
#include <algorithm>
#include <vector>

namespace dvc {

// Pinned staging of a batch call: kStageSlots slots of at most kStageSlot bytes
// in turn, whatever the batch's size.  The transfer over PCIe is several times
// faster than the copy between a slot and the caller's memory, so a few slots keep
// it ahead; all of a batch's bytes pinned at once, 0.9 MB a CIF pair of side
// information, grow with the caller's list and stay pinned afterwards.
constexpr size_t kStageSlot = 8u << 20;
constexpr int kStageSlots = 4;

// The pieces that the range [at[0], at[n]) is moved in, as part numbers: piece k
// holds the parts [cut[k], cut[k+1]), part i being [at[i], at[i+1]), n >= 1.  `want`
// pieces of like size, more where one would not fit a slot.  A part larger than a
// slot is a piece of its own.
inline std::vector<int> stage_pieces(const std::vector<size_t> &at, int want) {
  const int n = (int)at.size() - 1;
  const size_t share = (at[n] - at[0] + want - 1) / want;
  std::vector<int> cut{0};
  for (int i = 1; i < n; i++) {
    const size_t begin = at[cut.back()];
    if (at[i] - begin >= share || at[i + 1] - begin > kStageSlot) cut.push_back(i);
  }
  cut.push_back(n);
  return cut;
}

// Bytes of the largest piece.
inline size_t stage_slot_bytes(const std::vector<size_t> &at, const std::vector<int> &cut) {
  size_t m = 0;
  for (size_t k = 0; k + 1 < cut.size(); k++) m = std::max(m, at[cut[k + 1]] - at[cut[k]]);
  return m;
}

// Bytes that come back for one side-information request: a byte a pixel of side
// information and four each of residue and alpha, nothing of what it leaves out.
inline size_t si_result_bytes(size_t pixels, bool residue, bool alpha) {
  return pixels * (1 + (residue ? 4 : 0) + (alpha ? 4 : 0));
}

}  // namespace dvc
