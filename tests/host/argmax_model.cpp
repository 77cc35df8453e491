// The segment arg-max and the top-k built on it, run on the host: lanes as an
// array, each step of seg_argmax (smoe_common.hpp) as the lane permutation it
// is, select_key and argmax_take themselves compiled from the header.  Every
// lane must end with the same pair, and K rounds must take K distinct entries
// in the selection's order: values descending with NaN as +infinity, ties to
// the lowest index.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "smoe_common.hpp"

namespace {

constexpr int kNone = smoe::kWideBig;

int partner(int step, int l) {
  switch (step) {
    case 0: return l ^ 1;
    case 1: return l ^ 2;
    case 2: return (l & ~7) | (7 - (l & 7));
    case 3: return (l & ~15) | (15 - (l & 15));
    case 4: return l ^ 16;
    default: return l ^ 32;
  }
}

void seg_argmax(int seg, std::vector<float>& v, std::vector<int>& i) {
  const int steps = seg == 16 ? 4 : (seg == 32 ? 5 : 6);
  for (float& x : v) x = smoe::select_key(x);
  for (int s = 0; s < steps; ++s) {
    const std::vector<float> ov = v;
    const std::vector<int> oi = i;
    for (int l = 0; l < seg; ++l) smoe::argmax_take(v[l], i[l], ov[partner(s, l)], oi[partner(s, l)]);
  }
}

// Top-k of x (E entries, entry l + seg * c in lane l) as the routing kernels
// take it; false with a message where lanes disagree.
bool topk(int seg, const std::vector<float>& x, int K, std::vector<int>& out) {
  const int E = static_cast<int>(x.size()), V = (E + seg - 1) / seg;
  std::vector<char> sel(E, 0);
  out.clear();
  for (int j = 0; j < K; ++j) {
    std::vector<float> cv(seg, -INFINITY);
    std::vector<int> ci(seg, kNone);
    for (int l = 0; l < seg; ++l)
      for (int c = 0; c < V; ++c) {
        const int e = l + seg * c;
        const bool cand = e < E && !sel[e];
        smoe::argmax_take(cv[l], ci[l], cand ? smoe::select_key(x[e]) : -INFINITY, cand ? e : kNone);
      }
    seg_argmax(seg, cv, ci);
    for (int l = 1; l < seg; ++l)
      if (ci[l] != ci[0] || cv[l] != cv[0]) {
        std::printf("lanes disagree: seg %d E %d pick %d: lane 0 takes %d, lane %d takes %d\n", seg, E, j,
                    ci[0], l, ci[l]);
        return false;
      }
    if (ci[0] < 0 || ci[0] >= E || sel[ci[0]]) {
      std::printf("seg %d E %d pick %d: %d taken again or out of range\n", seg, E, j, ci[0]);
      return false;
    }
    sel[ci[0]] = 1;
    out.push_back(ci[0]);
  }
  return true;
}

}  // namespace

int main() {
  std::mt19937 rng(5);
  const float special[] = {NAN, -NAN, INFINITY, -INFINITY, 0.f, -0.f, 1.f, -1e4f};
  int runs = 0;
  for (const int E : {1, 3, 4, 8, 15, 16, 17, 31, 32, 33, 64, 65, 128, 200, 256})
    for (int rep = 0; rep < 400; ++rep) {
      const int seg = E <= 16 ? 16 : (E <= 32 ? 32 : 64);
      const int K = 1 + static_cast<int>(rng() % std::min(E, 16));
      const int odds = rep % 5;  // 0: finite only, 4: specials only
      std::vector<float> x(E);
      for (float& v : x)
        v = static_cast<int>(rng() % 4) < odds ? special[rng() % 8]
                                               : static_cast<float>(static_cast<int>(rng() % 41)) - 20.f;
      std::vector<int> got, want(E);
      if (!topk(seg, x, K, got)) return 1;
      for (int e = 0; e < E; ++e) want[e] = e;
      std::stable_sort(want.begin(), want.end(), [&](int a, int b) {
        return (std::isnan(x[a]) ? INFINITY : x[a]) > (std::isnan(x[b]) ? INFINITY : x[b]);
      });
      want.resize(K);
      if (got != want) {
        std::printf("E %d K %d rep %d: picks differ from the sorted order\n", E, K, rep);
        return 1;
      }
      ++runs;
    }
  std::printf("%d selections agree\n", runs);
  return 0;
}
