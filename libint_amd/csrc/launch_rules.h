// The rules by which launches are laid out, as plain functions of sizes (no
// HIP types: tests/test_plan_layout.py compiles them alone).
#pragma once
#include <algorithm>
#include <cstdint>
#include <numeric>
#include <vector>

namespace l2g_impl {

// Scratch doubles of the pieces of one ERI plan, over all its classes: 2 GiB,
// as much as the lane scratch of one heavy class on the per-lane kernels.
// 400,000 quartets of 58 s..f classes, K to 8, take 1.4 GB.
constexpr int64_t kPlanPieceDoubles = int64_t(1) << 28;

// A class whose primitive loops could be cut into pieces: scratch doubles of
// its pieces, and the time that they save (any unit).
struct PieceCandidate {
  int64_t doubles = 0;
  double gain = 0;
};

// Which of a plan's candidates are cut: by decreasing gain while their
// scratch fits `cap`; the others run unsplit.
inline std::vector<char> choose_pieces(const std::vector<PieceCandidate>& c, int64_t cap) {
  std::vector<size_t> order(c.size());
  std::iota(order.begin(), order.end(), size_t(0));
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return c[a].gain > c[b].gain; });
  std::vector<char> cut(c.size(), 0);
  for (size_t i : order)
    if (c[i].doubles <= cap) cut[i] = 1, cap -= c[i].doubles;
  return cut;
}

// Pieces of a shell pair's (p|p) loop of w primitive quartets for its Schwarz
// factor: 64 each, longer where one pair's would not fit a window of
// kSchwarzDoubles (a piece leaves `stride` of them).
constexpr int64_t kSchwarzPiece = 64, kSchwarzDoubles = int64_t(1) << 25;
inline int64_t schwarz_pieces(int64_t w, int64_t stride) {
  return std::max<int64_t>(1, std::min((w + kSchwarzPiece - 1) / kSchwarzPiece, kSchwarzDoubles / stride));
}

}  // namespace l2g_impl
