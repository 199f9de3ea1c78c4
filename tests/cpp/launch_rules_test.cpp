// The launch rules on the command line, for tests/test_plan_layout.py.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "launch_rules.h"

using namespace l2g_impl;

int main(int argc, char** argv) {
  if (argc >= 3 && !std::strcmp(argv[1], "pieces")) {  // cap, then doubles and gain of each class
    std::vector<PieceCandidate> c;
    for (int i = 3; i + 1 < argc; i += 2) c.push_back({std::atoll(argv[i]), std::atof(argv[i + 1])});
    const int64_t cap = std::atoll(argv[2]);
    for (char x : choose_pieces(c, cap ? cap : kPlanPieceDoubles)) std::printf("%d ", x);
    return 0;
  }
  if (argc == 4 && !std::strcmp(argv[1], "schwarz")) {
    std::printf("%lld %lld", (long long)schwarz_pieces(std::atoll(argv[2]), std::atoll(argv[3])), (long long)kSchwarzDoubles);
    return 0;
  }
  if (argc >= 4 && !std::strcmp(argv[1], "tiers")) {  // len, then the items' primitive quartets
    std::vector<int> w;
    for (int i = 3; i < argc; ++i) w.push_back(std::atoi(argv[i]));
    const LaneTiers t = lane_tiers(w.data(), (int64_t)w.size(), std::atoll(argv[2]));
    for (int x : t.n) std::printf("%d ", x);
    std::printf("%lld", (long long)t.units());
    return 0;
  }
  if (argc == 6 && !std::strcmp(argv[1], "length")) {
    std::printf("%lld", (long long)lane_length(std::atoi(argv[2]), std::atoll(argv[3]), std::atoll(argv[4]),
                                               std::atoi(argv[5]) != 0));
    return 0;
  }
  if (argc == 11 && !std::strcmp(argv[1], "faster")) {  // LaneCost, then quartets, primitive quartets, the deepest's
    float c[6];
    for (int i = 0; i < 6; ++i) c[i] = (float)std::atof(argv[2 + i]);
    const LaneCost k{c[0], c[1], c[2], c[3], c[4], c[5]};
    std::printf("%d %d", lane_faster(k, std::atoll(argv[8]), std::atoll(argv[9]), std::atoll(argv[10])), lane_always(k));
    return 0;
  }
  if (argc == 5 && !std::strcmp(argv[1], "unsplit")) {
    std::printf("%d", unsplit_generic(std::atoll(argv[2]), std::atoll(argv[3]), std::atoll(argv[4]), 256));
    return 0;
  }
  return 1;
}
