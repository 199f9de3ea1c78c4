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
  return 1;
}
