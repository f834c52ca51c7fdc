// Writes attention plans as the plan kernel does and walks them as the
// attention kernels do (csrc/attn_plan.h), for calls of fewer and of more
// tokens than the plan was made for, buffers of zeros and of noise: every walk
// ends, takes each token once, and follows the plan's segments where the plan
// knows the tokens.
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "attn_plan.h"

using namespace fr;

static int walk(const int32_t* rec, int ntok, std::vector<int>& first) {
  int steps = 0, at = 0;
  first.clear();
  for (; at < ntok && steps <= ntok; ++steps) {
    first.push_back(at);
    at += plan_count(rec[kPlanCount + at], at, ntok);
  }
  return at == ntok ? steps : -1;
}

int main() {
  std::mt19937 rng(7);
  long walks = 0;
  for (int tok : {4, 8, 16, 32}) {
    const int stride = plan_stride(tok);
    for (int round = 0; round < 400; ++round) {
      const int T = 1 + rng() % (5 * tok), groups = (T + tok - 1) / tok;
      std::vector<int32_t> plan(size_t(groups) * stride, round % 3 == 0 ? int32_t(rng()) : 0);
      std::vector<std::vector<int>> starts(groups);
      for (int g = 0; g < groups; ++g) {
        const int ntok = T - g * tok < tok ? T - g * tok : tok;
        int32_t* rec = plan.data() + int64_t(g) * stride;
        rec[kPlanTag] = plan_tag(g);
        for (int i = 0; i < tok; ++i) rec[kPlanCount + i] = rec[plan_shared_at(tok) + i] = 0;
        for (int at = 0; at < ntok;) {
          const int n = 1 + rng() % (ntok - at);
          starts[g].push_back(at);
          rec[kPlanCount + at] = n;
          rec[plan_shared_at(tok) + at] = 100 * g + at;
          at += n;
        }
      }
      // read by a call of any number of tokens up to whole groups
      for (int reader = 1; reader <= groups * tok; ++reader)
        for (int g = 0; g * tok < reader; ++g) {
          const int ntok = reader - g * tok < tok ? reader - g * tok : tok;
          const int32_t* rec = plan.data() + int64_t(g) * stride;
          std::vector<int> got, want;
          if (rec[kPlanTag] != plan_tag(g) || walk(rec, ntok, got) < 0) return std::printf("walk %d %d\n", T, reader), 1;
          const int known = T - g * tok < ntok ? T - g * tok : ntok;
          for (int s : starts[g])
            if (s < known) want.push_back(s);
          for (int s = known; s < ntok; ++s) want.push_back(s);  // unknown to the plan: one by one
          if (got != want) return std::printf("segments %d %d %d\n", tok, T, reader), 1;
          ++walks;
        }
    }
    // no plan at all: the tag says so; a walk over zeros or noise ends all the same
    for (int round = 0; round < 2000; ++round) {
      std::vector<int32_t> rec(stride, 0);
      if (round)
        for (int32_t& x : rec) x = int32_t(rng());
      std::vector<int> got;
      if (!round && rec[kPlanTag] == plan_tag(0)) return std::printf("tag\n"), 1;
      for (int ntok = 1; ntok <= tok; ++ntok)
        if (walk(rec.data(), ntok, got) < 0) return std::printf("noise %d\n", ntok), 1;
    }
  }
  std::printf("walks=%ld\n", walks);
  return 0;
}
