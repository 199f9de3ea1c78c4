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

// Lanes per item of a per-lane ERI launch: items at the front of the list (w,
// decreasing: their primitive quartets) with 64, 16, 4 lanes and one lane
// each.  An item shares its loop between lanes from `len` primitive quartets
// on, and none is walked for much longer than that.
struct LaneTiers {
  int n[4] = {0, 0, 0, 0};
  int64_t units() const { return n[0] + (n[1] + 3) / 4 + (n[2] + 15) / 16 + (n[3] + 63) / 64; }
  bool operator==(const LaneTiers& o) const { return std::equal(n, n + 4, o.n); }
};
inline LaneTiers lane_tiers(const int* w, int64_t n, int64_t len) {
  auto upto = [&](int64_t least) {  // items of at least that many
    return (int)(std::partition_point(w, w + n, [&](int x) { return x >= least; }) - w);
  };
  const int a = upto(32 * len), b = upto(4 * len), c = upto(len);
  LaneTiers t;
  t.n[0] = a, t.n[1] = b - a, t.n[2] = c - b, t.n[3] = (int)n - c;
  return t;
}

// That length.  Summing a group's accumulators (`targets`) costs classes of
// many of them more than a short loop: 3000 quartets of 256 primitive quartets
// take 38 us at 8 and 41 at 16 in (ps|ps), 84 and 86 in (pp|pp), where 20,000
// of 16 take 98 and 80.  A launch that fills the chip anyway shares less: half
// of a lane's share of the class (`lanes`: the chip's, one wave per SIMD) is
// not cut ((pp|pp), 150,000 of 256: 1252 us, 1970 with sharing from 16 on),
// unless the sums are short ((ps|ps): 350 us with sharing, 490 without).
// Not by_batch: by the class alone, so that a quartet's bits do not depend on
// the other quartets.
inline int64_t lane_length(int targets, int64_t nprim, int64_t lanes, bool by_batch) {
  const int64_t base = targets <= 32 ? 8 : 16;
  return by_batch && targets > 24 ? std::max(base, nprim / (2 * lanes)) : base;
}

// ERI classes that have a per-lane kernel (codegen/gen_eri.py) besides their
// Rys kernel, with the measured costs of both (gen_rys.py, LANE_COST).
struct LaneCost {
  float lane_q, lane_p;   // ns per quartet and per primitive quartet on the per-lane kernel, with the chip full
  float rys_q, rys_p;     // the same on the Rys kernel
  float shallow, deep;    // us that a launch of few quartets takes longer on the per-lane kernel: 1, many primitives
};

// On the per-lane kernel whatever the batch: the rule for single quartets and
// with the split off, where a quartet's kernel may not depend on the others.
// These classes are slower there in one place, (ps|pp) quartets of 1
// primitive quartet, 150,000 of them (75 against 64 us).
inline bool lane_always(const LaneCost& c) { return c.lane_p > 0 && c.shallow <= 1 && c.deep <= 1; }

// Whether n quartets of nprim primitive quartets in all, wmax at most, are
// faster on the per-lane kernel, by 5 % at least: the two lines cross at a few
// thousand to some ten thousand quartets of 50 to 256 primitive quartets in
// the heavier classes ((pp|pp), 256: 86 against 82 us at 3000, 611 against 991
// at 60,000), and those of 1 primitive quartet stay on the Rys kernel
// (150,000: 174 against 92 us).
inline bool lane_faster(const LaneCost& c, int64_t n, int64_t nprim, int64_t wmax) {
  if (!(c.lane_p > 0)) return false;
  const double lane = 1e3 * (wmax >= 16 ? c.deep : c.shallow) + (double)c.lane_q * n + (double)c.lane_p * nprim;
  return lane < 0.95 * ((double)c.rys_q * n + (double)c.rys_p * nprim);
}

// Layout off, classes of so large a block that few of a Rys kernel's slots
// share a deep quartet ((df|ff) and (ff|ff): 3): a quartet's loop takes 0.8 to
// 1.5 us a primitive quartet there, the generic kernel, which cuts it, 0.6 to
// 1.4 ms and 0.045 to 0.075 us a primitive quartet of the class.  One quartet
// of 4096 among 99 of 1: (df|ff) 3.4 against 0.74 ms, (ff|ff) 6.1 against 1.7;
// 60 of them 3.5 against 11.9 ms.
inline bool unsplit_generic(int64_t count, int64_t nprim, int64_t wmax, int64_t ncu) {
  return count <= 16 * ncu && wmax > 1000 + nprim / 18;
}

// Pieces of a shell pair's (p|p) loop of w primitive quartets for its Schwarz
// factor: 64 each, longer where one pair's would not fit a window of
// kSchwarzDoubles (a piece leaves `stride` of them).
constexpr int64_t kSchwarzPiece = 64, kSchwarzDoubles = int64_t(1) << 25;
inline int64_t schwarz_pieces(int64_t w, int64_t stride) {
  return std::max<int64_t>(1, std::min((w + kSchwarzPiece - 1) / kSchwarzPiece, kSchwarzDoubles / stride));
}

}  // namespace l2g_impl
