// Every interleaving of page_claim (fragpack_amd/csrc/fp_page_claim.hpp) for a
// few records of one page.  A record is re-run from its start with the results
// its atomics have had so far; the first atomic past them is its next step.
//
//   page_claim_model PAGE FILL POLLS NEED...   (POLLS 0: as the encoder's, and
//   a poll that would see the same fill again waits for a change)
//
// Prints "ok STATES" or the first violation: records that overlap or leave the
// page, a fill that is not what the placed records make it, a spilled record
// that fits what is left, records that wait for ever.
#define __host__
#define __device__
#include "../fragpack_amd/csrc/fp_page_claim.hpp"

#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

namespace {

struct Op {
  char kind;
  int a, b;
};

struct Replay {
  const std::vector<int>& seen;
  size_t at = 0;
  int next(Op op) {
    if (at < seen.size()) return seen[at++];
    throw op;
  }
  int add(int n) { return next({'a', n, 0}); }
  int sub(int n) { return next({'s', n, 0}); }
  int load() { return next({'l', 0, 0}); }
  int cas(int from, int to) { return next({'c', from, to}); }
};

struct Search {
  int page, start, polls;
  std::vector<int> needs;
  std::set<std::vector<int>> seen;
  const char* bad = nullptr;

  // the record's next atomic, or its place in ``off``
  bool step(int need, const std::vector<int>& hist, Op& op, int& off) const {
    Replay r{hist};
    int left = polls ? polls : fp::kPageWaitPolls;
    try {
      off = fp::page_claim(r, r.add(need), need, page, left);
      return false;
    } catch (const Op& next) {
      op = next;
      return true;
    }
  }

  void run(int fill, std::vector<std::vector<int>>& hist) {
    if (bad) return;
    std::vector<int> key{fill};
    for (auto& h : hist) {
      key.push_back(-1 - (int)h.size());
      key.insert(key.end(), h.begin(), h.end());
    }
    if (!seen.insert(key).second) return;
    const int n = (int)needs.size();
    std::vector<int> offs(n, -2);
    bool moved = false, done = true;
    for (int i = 0; i < n; ++i) {
      Op op{};
      if (!step(needs[i], hist[i], op, offs[i])) continue;
      done = false;
      offs[i] = -2;
      if (op.kind == 'l' && !polls && hist[i].size() > 2 && hist[i].back() == fill) continue;  // sees nothing new
      moved = true;
      int after = fill;
      if (op.kind == 'a') after = fill + op.a;
      if (op.kind == 's') after = fill - op.a;
      if (op.kind == 'c' && fill == op.a) after = op.b;
      hist[i].push_back(fill);
      run(after, hist);
      hist[i].pop_back();
      if (bad) return;
    }
    if (!done && !moved) bad = "records wait for ever";
    if (!done) return;
    int sum = start;
    for (int i = 0; i < n; ++i) {
      if (offs[i] < 0) continue;
      sum += needs[i];
      if (offs[i] < start || offs[i] + needs[i] > page) bad = "a record lies outside the page";
      for (int j = 0; j < i; ++j)
        if (offs[j] >= 0 && offs[i] < offs[j] + needs[j] && offs[j] < offs[i] + needs[i]) bad = "records overlap";
    }
    if (fill != sum) bad = "the fill is not what the placed records make it";
    for (int i = 0; i < n; ++i)
      if (offs[i] == -1 && sum + needs[i] <= page && !polls) bad = "a spilled record fits what is left";
  }
};

}  // namespace

int main(int argc, char** argv) {
  if (argc < 5) return 2;
  Search s{atoi(argv[1]), atoi(argv[2]), atoi(argv[3]), {}, {}, nullptr};
  for (int i = 4; i < argc; ++i) s.needs.push_back(atoi(argv[i]));
  std::vector<std::vector<int>> hist(s.needs.size());
  s.run(s.start, hist);
  if (s.bad) {
    printf("%s\n", s.bad);
    return 1;
  }
  printf("ok %zu\n", s.seen.size());
  return 0;
}
